"""The fused move of few electrons with its pending record in LDS
(k_move_small): electrons up to the lane group's width, one or several passes
over the centres' basis functions, both movers, more occupied orbitals than
its matrix tiles take, the last block partly empty.
Against k_ratio_1e (QMCW_NO_MOVE_SMALL), whose operations it repeats up to
the order of a matrix product's sums: identical decisions, local energies to
1e-10."""
import dataclasses

import numpy as np
import pytest

import oracle
from champ_amd import rng, system
from champ_amd.engine import Engine

pytestmark = pytest.mark.gpu


def _system(name):
    if name == "c2":
        return system.c2_dimer(2)
    if name == "be":
        return system.be_atom(1)
    n, m = name
    s = system.random_molecule(400 + n, nelec=max(n, 2), ncent=m, zeff=6.0)
    if n == 1:                         # one electron, no down spin
        s.nelec, s.nup = 1, 1
        s.det_up, s.det_dn = s.det_up[:, :1], s.det_dn[:, :0]
    return s


def _walk(s, W, G, prec="fp64", imetro=1, nst=2):
    x = system.random_walkers(s, W, seed=31)
    seeds = np.asarray(rng.walker_seeds("1837465927472523", W), np.int32)
    e = Engine(s, W, prec)
    e.set_group_width(G)
    e.set_vmc_mover(imetro)
    e.set_walkers(x)
    e.set_rng(seeds)
    r = e.vmc(nst, delta=0.4)
    out = (e.get_walkers(), r["naccept"], r["eloc"], e.get_rng())
    e.close()
    return x, seeds, out


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("name,G,imetro", [("c2", 8, 1), ("c2", 16, 6), ("be", 8, 6), ((1, 1), 8, 1),
                                           ((2, 1), 16, 1), ((5, 2), 8, 6), ((8, 3), 8, 1), ((9, 4), 16, 1),
                                           ((15, 2), 16, 6), ((16, 5), 16, 1), ((17, 5), 32, 1)], ids=str)
def test_equals_the_general_kernel(monkeypatch, name, G, imetro, prec):
    s = _system(name)
    a = _walk(s, 19, G, prec, imetro)[2]
    monkeypatch.setenv("QMCW_NO_MOVE_SMALL", "1")
    b = _walk(s, 19, G, prec, imetro)[2]
    assert np.array_equal(a[1], b[1]) and np.array_equal(a[3], b[3])
    if imetro == 1:                    # the proposal takes no velocity: the same numbers
        assert np.array_equal(a[0], b[0])
    else:
        # the drift carries the velocity's rounding, 1e-7 (1e-15) of O(10) in
        # steps of O(1), through two steps
        assert np.max(np.abs(a[0] - b[0])) < (1e-11 if prec == "fp64" else 1e-5)
    tol, floor = (1e-10, 1e-8) if prec == "fp64" else (1e-4, 10.0)
    assert np.max(np.abs(a[2] - b[2]) / (np.abs(b[2]) + floor)) < tol



@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("name,G", [("c2", 8), ((8, 3), 8), ((15, 6), 16)], ids=str)
def test_passes_over_the_centres(monkeypatch, name, G, prec):
    """So many walkers that a block's LDS does not hold all basis values at
    once (20 and 10 blocks to a compute unit): one centre a pass with two and
    three centres, two centres a pass with six."""
    s = _system(name)
    W = 20011
    a = _walk(s, W, G, prec)[2]
    monkeypatch.setenv("QMCW_NO_MOVE_SMALL", "1")
    b = _walk(s, W, G, prec)[2]
    same = np.all(a[0] == b[0], axis=(1, 2)) & (a[1] == b[1])
    # FP32 rows in another order: a decision turns where the ratio lies within
    # some 1e-6 of the draw, up to 30 decisions a walker
    assert same.all() if prec == "fp64" else same.sum() >= W - 20
    assert np.array_equal(a[3][same], b[3][same])
    tol, floor = (1e-10, 1.0) if prec == "fp64" else (1e-3, 10.0)
    assert np.max((np.abs(a[2] - b[2]) / (np.abs(b[2]) + floor))[:, same]) < tol


@pytest.mark.parametrize("G", [8, 16])
@pytest.mark.parametrize("nvirt", [14, 32])
def test_more_orbitals_than_tiles(monkeypatch, G, nvirt):
    """18 and 36 occupied orbitals of a spin: beyond 16 at 8 lanes and 32 at
    16 the orbitals are taken one per lane."""
    s = system.c2_dimer(2)
    ref, exc = [0, 1, 2, 3], [[0, 1, 2, a] for a in range(4, 4 + nvirt)]
    n = 1 + 2 * nvirt
    g = np.random.default_rng(nvirt)
    s = dataclasses.replace(s, det_up=np.array([ref] + exc + [ref] * nvirt, np.int32),
                            det_dn=np.array([ref] + [ref] * nvirt + exc, np.int32),
                            csf_coef=np.concatenate([[1.0], g.normal(0, 0.1, n - 1)]),
                            csf_det_off=np.arange(n + 1, dtype=np.int32), csf_det=np.arange(n, dtype=np.int32),
                            csf_det_coef=np.ones(n))
    x, seeds, a = _walk(s, 19, G)
    o = oracle.Oracle(s).vmc_run(x, seeds, 2, 0.4)
    monkeypatch.setenv("QMCW_NO_MOVE_SMALL", "1")
    b = _walk(s, 19, G)[2]
    for r in (b[:2], (o["x"], o["naccept"])):
        assert np.array_equal(a[0], r[0]) and np.array_equal(a[1], r[1])
    assert np.array_equal(a[3], b[3]) and np.array_equal(a[3], o["rng"])
    assert np.max(np.abs(a[2] - b[2]) / (np.abs(b[2]) + 1e-8)) < 1e-10
    assert np.max(np.abs(a[2] - o["eloc"]) / (np.abs(o["eloc"]) + 1e-8)) < 1e-9
