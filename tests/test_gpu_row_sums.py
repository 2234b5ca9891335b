"""One-electron ratios whose e-e-n terms are summed over the centres before
they meet the pair's power of the distance (jas_pair_sum), at the number of
centres where FP64 starts to use it and about it, at both lane-group widths
and every order; walks against the oracle's (identical decisions, local
energies to 1e-9), and mixed precision, which always uses it."""
import numpy as np
import pytest

import oracle
from champ_amd import rng, system
from champ_amd.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("M,nordc,G", [(7, 4, 32), (8, 4, 32), (9, 4, 64), (8, 4, 16), (8, 2, 32), (8, 3, 64),
                                       (8, 5, 32), (8, 6, 64), (8, 7, 32), (1, 4, 32),
                                       (13, 4, 64), (14, 4, 32), (14, 4, 64), (15, 4, 32), (14, 4, 16), (14, 2, 32),
                                       (14, 3, 64), (14, 5, 32), (14, 6, 64), (14, 7, 32)])
def test_walks_match_oracle(M, nordc, G, prec):
    s = system.random_molecule(700 + M, nelec=21, ncent=M, zeff=4.0)
    g = np.random.default_rng(nordc)
    if nordc != s.nordc:
        nct = s.c.shape[0]
        s.nordc = nordc
        s.c = system.cusp_exact(g.normal(0, 0.02, (nct, system.nterms4(nordc))), nordc)
    W, nst = 5, 2
    x = system.random_walkers(s, W, seed=M)
    seeds = np.asarray(rng.walker_seeds("1837465927472523", W), np.int32)
    e = Engine(s, W, prec)
    e.set_group_width(G)
    e.set_walkers(x)
    e.set_rng(seeds)
    r = e.vmc(nst, delta=0.4)
    o = oracle.Oracle(s).vmc_run(x, seeds, nst, 0.4)
    if prec == "fp64":
        assert np.array_equal(e.get_walkers(), o["x"]) and np.array_equal(r["naccept"], o["naccept"])
        assert np.max(np.abs(r["eloc"] - o["eloc"]) / (np.abs(o["eloc"]) + 1e-8)) < 1e-9
    else:
        # FP32 factors of O(1) in 21 x M sums of 1e-7 rounding each; decisions
        # flip only where the ratio lies within 1e-5 of the draw
        same = np.all(e.get_walkers() == o["x"], axis=tuple(range(1, o["x"].ndim)))
        assert same.sum() >= W - 1
        # kinetic and potential terms of O(100) cancel in the local energy
        assert np.max((np.abs(r["eloc"] - o["eloc"]) / (np.abs(o["eloc"]) + 10.0))[:, same]) < 1e-3
    e.close()
