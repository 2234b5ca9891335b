"""The fused move of few electrons with its pending record in LDS
(k_move_small): electrons up to the lane group's width, one or several passes
over the centres' basis functions, both movers, the last block partly empty.
Against k_ratio_1e (QMCW_NO_MOVE_SMALL), whose operations it repeats up to
the order of a matrix product's sums: identical decisions, local energies to
1e-10."""
import numpy as np
import pytest

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

