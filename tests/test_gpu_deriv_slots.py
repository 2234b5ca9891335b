"""The derivatives' slot sums (k_deriv_jas, k_deriv_nlpp) and assembly
(k_derivs) where their loops end: electrons about the lane-group widths,
centres whose shells take one or several passes of the basis tile, no pair
in range, every order of the e-e-n polynomial, one or two e-e coefficient
sets; lane-group and tile pseudopotentials.  Against the oracle with the
bounds of tests/test_gpu_derivs.py."""
import numpy as np
import pytest

import oracle
from champ_amd import system
from champ_amd.engine import Engine

pytestmark = pytest.mark.gpu


def _mol(nelec, ncent, nordc=4, nspin2b=1, big=False):
    s = system.random_molecule(500 + nelec, nelec=nelec, ncent=ncent, zeff=6.0, big_basis=big)
    g = np.random.default_rng(nordc)
    if nordc != s.nordc:
        s.nordc = nordc
        s.c = (system.cusp_exact(g.normal(0, 0.03, (3, system.nterms4(nordc))), nordc)
               if nordc > 1 else np.zeros((3, 0)))
    if nspin2b == 2:
        s.nspin2b = 2
        s.b = np.concatenate([s.b, s.b * 0.9])
        s.b[1, 0] = 0.25
    return system.molecule_derivs(s)


CASES = [(2, 1, 4, 1, False), (7, 2, 4, 2, False), (8, 3, 4, 1, False), (9, 2, 4, 1, True),
         (16, 3, 4, 1, False), (17, 2, 4, 2, False), (32, 2, 4, 1, False), (33, 3, 4, 1, True),
         (6, 2, 2, 1, False), (6, 2, 3, 1, False), (6, 2, 5, 1, False), (6, 2, 6, 1, False),
         (6, 2, 7, 1, False)]


@pytest.mark.parametrize("nelec,ncent,nordc,nspin2b,big", CASES)
@pytest.mark.parametrize("tiles", ["0", "2"])
def test_derivs_match_oracle(monkeypatch, nelec, ncent, nordc, nspin2b, big, tiles):
    monkeypatch.setenv("QMCW_NLPP_TILES", tiles)
    s = _mol(nelec, ncent, nordc, nspin2b, big)
    W = 9
    x = system.random_walkers(s, W, seed=nelec)
    x[0] += 1.5                        # few pairs in range or none
    r = oracle.Oracle(s).eval_batch(x, derivs=True)
    for G in (8, 64) if nelec < 17 else (32,):
        e = Engine(s, W)
        e.set_group_width(G)
        e.set_walkers(x)
        dp, de = e.derivs()
        assert np.max(np.abs(dp - r["dpsi"]) / (np.abs(r["dpsi"]) + 1e-9)) < 1e-9
        assert np.max(np.abs(de - r["deloc"]) / (np.abs(r["deloc"]) + 1e-8)) < 1e-8
        e.close()
