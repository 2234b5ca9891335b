"""The one-electron move at 32 and 64 lanes about the orbital counts where its
lanes share the basis (a half and a quarter of the width), with basis sizes
that leave remainders in the batched sums and Slater updates; walks against
the oracle's (identical decisions, local energies to 1e-9), and the split
launches of the same move."""
import numpy as np
import pytest

import oracle
from champ_amd import rng, system
from champ_amd.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("split", ["0", "1"])
@pytest.mark.parametrize("nelec,G", [(15, 32), (16, 32), (18, 32), (31, 32), (34, 32), (32, 64), (34, 64),
                                     (63, 64), (66, 64)])
def test_walks_match_oracle(monkeypatch, nelec, G, split):
    monkeypatch.setenv("QMCW_SPLIT_MOVE", split)
    s = system.random_molecule(800 + nelec, nelec=nelec, ncent=4 + nelec // 8, zeff=4.0)
    W, nst = 3, 1
    x = system.random_walkers(s, W, seed=nelec)
    seeds = np.asarray(rng.walker_seeds("1837465927472523", W), np.int32)
    e = Engine(s, W)
    e.set_group_width(G)
    e.set_walkers(x)
    e.set_rng(seeds)
    r = e.vmc(nst, delta=0.4)
    o = oracle.Oracle(s).vmc_run(x, seeds, nst, 0.4)
    assert np.array_equal(e.get_walkers(), o["x"]) and np.array_equal(r["naccept"], o["naccept"])
    assert np.max(np.abs(r["eloc"] - o["eloc"]) / (np.abs(o["eloc"]) + 1e-8)) < 1e-9
    e.close()
