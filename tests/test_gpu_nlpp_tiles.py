"""The pseudopotential with its points' Jastrow on MFMA (k_full_nlpp_tiles)
at the sizes where its tiles end: electrons about the 16-column tiles and the
passes of three and four of them, centres about the steps of four, one to
four wavefronts per walker, every order of the e-e-n polynomial, g and h
shells.  FP64 against the oracle (bounds of the molecules' parity tests);
mixed against the lane-group kernel of the same precision, whose FP32 sums
run in another order (2^-24 per operation over the few thousand terms of a
point's Jastrow, times |V_nl| of a few Ha, stays below 1e-4)."""
import dataclasses
import os
import sys

import numpy as np
import pytest

import oracle
from champ_amd import system
from champ_amd.engine import Engine

sys.path.insert(0, os.path.dirname(__file__))
pytestmark = pytest.mark.gpu


def _mol(nelec, ncent, nordc=4, gh=False):
    s = system.random_molecule(300 + nelec, nelec=nelec, ncent=ncent, zeff=6.0, gh_shells=gh)
    if nordc != s.nordc:
        g = np.random.default_rng(nordc)
        s.nordc = nordc
        s.c = system.cusp_exact(g.normal(0, 0.03, (3, system.nterms4(nordc))), nordc)
    return s


CASES = [(2, 1, 4, False), (15, 3, 4, False), (16, 4, 4, False), (17, 5, 4, True),
         (33, 2, 4, False), (48, 3, 4, False), (49, 4, 4, False), (65, 6, 4, False),
         (9, 3, 2, False), (9, 3, 3, False), (18, 3, 5, False), (9, 3, 6, False), (9, 3, 7, False)]


@pytest.mark.parametrize("nelec,ncent,nordc,gh", CASES)
@pytest.mark.parametrize("waves", [1, 2, 4])
def test_tiles_match_oracle(monkeypatch, nelec, ncent, nordc, gh, waves):
    monkeypatch.setenv("QMCW_NLPP_TILES", str(waves))
    s = _mol(nelec, ncent, nordc, gh)
    W = 5
    x = system.random_walkers(s, W, seed=nelec)
    x[0] += 2.0                        # a walker with few pairs in range or none
    e = Engine(s, W)
    e.set_walkers(x)
    g = e.psi_at()
    o9 = oracle.Oracle(s).eval_batch(x)["out9"]
    assert np.max(np.abs(g["epot"] - o9[:, 4]) / (np.abs(o9[:, 4]) + 1e-8)) < 1e-9


@pytest.mark.parametrize("nelec,ncent", [(8, 3), (33, 4), (65, 6)])
def test_mixed_tiles_match_lane_groups(monkeypatch, nelec, ncent):
    s = _mol(nelec, ncent)
    x = system.random_walkers(s, 24, seed=5)
    out = []
    for tiles in ("0", "2"):
        monkeypatch.setenv("QMCW_NLPP_TILES", tiles)
        e = Engine(s, 24, "mixed")
        e.set_walkers(x)
        out.append(e.psi_at()["epot"])
        e.close()
    scale = np.abs(out[0]) + 1.0
    assert np.median(np.abs(out[0] - out[1]) / scale) < 1e-5
    assert np.max(np.abs(out[0] - out[1]) / scale) < 1e-3


@pytest.mark.parametrize("tmoves", [0, 1])
def test_dmc_generations_on_tiles(monkeypatch, tmoves):
    from test_gpu_dmc import test_dmc_generations_match_oracle
    monkeypatch.setenv("QMCW_NLPP_TILES", "2")
    test_dmc_generations_match_oracle("c2_dimer", 0.3, tmoves)


def test_batch_of_tiles(monkeypatch):
    """One launch sequence with every pseudopotential on tiles (by the rule,
    test_gpu_batch.py has systems on either side of it)."""
    from test_gpu_batch import test_one_launch_batch_matches_oracle
    monkeypatch.setenv("QMCW_NLPP_TILES", "4")
    test_one_launch_batch_matches_oracle(monkeypatch, "0")


@pytest.mark.parametrize("ncent", [1600, 2900])
def test_pair_flags_beyond_the_lds(monkeypatch, ncent):
    """256 electrons: the flags of 410,000 pairs take 77 KB of a block's
    160 KB of LDS, those of 742,000 would take 139 KB beside the tiles' own 26
    and stay in lane groups.  Against the lane groups, whose FP64 sums run in
    another order."""
    s = system.random_molecule(12, nelec=2, ncent=1, zeff=4.0)
    side = int(np.ceil(ncent ** (1 / 3)))
    grid = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3)[:ncent] * 2.5
    g = np.random.default_rng(2)
    types = np.where(np.arange(ncent) < 128, 1, 0).astype(np.int32)
    nb = int(np.diff(s.ctype_bas_off)[types].sum())
    s = dataclasses.replace(s, nelec=256, nup=128, cent=grid, iwctype=types,
                            coef=g.normal(0.0, 0.3, (128, nb)), det_up=np.arange(128, dtype=np.int32)[None],
                            det_dn=np.arange(128, dtype=np.int32)[None])
    x = system.random_walkers(s, 1, seed=9, sigma=0.5)
    out = []
    for tiles in ("0", "4"):
        monkeypatch.setenv("QMCW_NLPP_TILES", tiles)
        e = Engine(s, 1)
        e.set_walkers(x)
        out.append(e.psi_at()["epot"][0])
        e.close()
    assert np.isfinite(out[0]) and abs(out[1] - out[0]) < 1e-9 * abs(out[0])
