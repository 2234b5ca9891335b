"""Determinants of small spins in LDS (k_det_small): spins of up to 15
electrons, also empty ones, single and multiple determinants, the last block
partly empty.  Walks against the oracle's (identical decisions, local
energies to 1e-9) and against k_full_det (QMCW_NO_DET_SMALL), whose
operations it repeats (1e-10); 16 electrons of a spin stay there."""
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


@pytest.mark.parametrize("name", ["c2", "be", (1, 1), (2, 1), (5, 2), (8, 3), (9, 4), (15, 2), (16, 5)],
                         ids=str)
@pytest.mark.parametrize("G", [8, 16])
def test_small_walks_match_oracle(name, G):
    s = _system(name)
    if s.nelec > G:
        pytest.skip("more electrons than lanes")
    W = 19                             # the last group partly empty
    x, seeds, (xs, nacc, eloc, rs) = _walk(s, W, G)
    o = oracle.Oracle(s).vmc_run(x, seeds, 2, 0.4)
    assert np.array_equal(xs, o["x"]) and np.array_equal(nacc, o["naccept"])
    assert np.array_equal(rs, o["rng"])
    assert np.max(np.abs(eloc - o["eloc"]) / (np.abs(o["eloc"]) + 1e-8)) < 1e-9


@pytest.mark.parametrize("name,imetro", [("c2", 1), ("be", 6), ((9, 4), 1), ((24, 4), 1), ((31, 3), 1)], ids=str)
def test_equals_the_general_kernel(monkeypatch, name, imetro):
    s = _system(name)
    G = 8 if s.nelec <= 8 else 16 if s.nelec <= 16 else 32
    a = _walk(s, 11, G, imetro=imetro)[2]
    monkeypatch.setenv("QMCW_NO_DET_SMALL", "1")
    b = _walk(s, 11, G, imetro=imetro)[2]
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]) and np.array_equal(a[3], b[3])
    assert np.max(np.abs(a[2] - b[2]) / (np.abs(b[2]) + 1e-8)) < 1e-10


def test_small_walks_with_reinversion_and_mixed():
    s = system.c2_dimer(2)
    x, seeds, a = _walk(s, 13, 8)
    e = Engine(s, 13)
    e.set_group_width(8)
    e.set_walkers(x)
    e.set_rng(seeds)
    e.set_reinversion(3)
    e.vmc_device(2, 0.4)
    assert np.array_equal(e.get_walkers(), a[0])
    e.close()
    m = _walk(s, 13, 8, "mixed")[2]
    assert np.median(np.abs(m[2] - a[2])) < 1e-4
