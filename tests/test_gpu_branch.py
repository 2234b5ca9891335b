"""The device split_join (k_split_join, the branching qmcw_dmc_step runs)
against the host routine qmcw_split_join -- itself bit-exact against the
reference's split_join (tests/test_branch_ref.py) -- on the same 70 weight
vectors: identical weights, copies, streams, populations, branching counts
and branching stream.  The DMC generations of tests/test_gpu_dmc.py run the
device path against the oracle; one of them is repeated on the host path."""
import ctypes as C
import os
import sys

import numpy as np
import pytest

from champ_amd import abi

sys.path.insert(0, os.path.dirname(__file__))
from test_branch_ref import _cases  # noqa: E402

pytestmark = pytest.mark.gpu
_pd, _pi = C.POINTER(C.c_double), C.POINTER(C.c_int32)


def _run(fn, w, cap, brng, rng):
    wt = np.zeros(cap)
    wt[:len(w)] = w
    origin = np.zeros(cap, np.int32)
    r = np.array(rng, np.int32).copy()
    b = np.array(brng, np.int32).copy()
    n, nb = C.c_int32(), C.c_int32()
    st = fn(len(w), cap, wt.ctypes.data_as(_pd), origin.ctypes.data_as(_pi), r.ctypes.data_as(_pi),
            b.ctypes.data_as(_pi), C.byref(n), C.byref(nb))
    k = n.value
    return st, (wt[:k], origin[:k], r[:k], b, k, nb.value)


def test_device_split_join_matches_host_routine():
    lib = abi.load_library()
    nsplit = 0
    for k, (w, cap) in enumerate(_cases()):
        b = [(17 * k + 5) % 4096, (311 * k + 9) % 4096, (1001 * k + 3) % 4096, (2 * k + 1) % 4096]
        rng = np.arange(4 * cap, dtype=np.int32).reshape(cap, 4) % 4096
        sh, h = _run(lib.qmcw_split_join, w, cap, b, rng)
        sg, g = _run(lib.qmcw_split_join_gpu, w, cap, b, rng)
        assert sh == 0 and sg == 0, (w, cap)
        for a, c in zip(h, g):
            assert np.array_equal(np.asarray(a), np.asarray(c)), (w, cap)
        nsplit += int(h[4] > len(w) - sum(1 for v in w if v == 0))
    assert nsplit > 5


# populations about the 4,096 walkers whose marks one pass of the kernel keeps,
# with room (no sort of the weights) and near the capacity (sorted), and
# weights that leave holes after the splits (compaction) or need them all
@pytest.mark.parametrize("n", [0, 1, 63, 64, 65, 4095, 4096, 4097, 8193])
@pytest.mark.parametrize("room", [0, 3, None])
@pytest.mark.parametrize("spread", [0.4, 1.2, 2.2])
def test_device_split_join_at_chunk_edges(n, room, spread):
    lib = abi.load_library()
    g = np.random.default_rng(n + int(10 * spread))
    w = np.exp(g.normal(0.0, spread, n))
    w[g.random(n) < 0.05] = 0.0
    if spread > 2:
        w[g.random(n) < 0.3] *= 0.01
    cap = max(1, 2 * n if room is None else n + room)
    rng = g.integers(0, 4096, (cap, 4), dtype=np.int32)
    sh, h = _run(lib.qmcw_split_join, w, cap, [7, 11, 13, 17], rng)
    sg, gp = _run(lib.qmcw_split_join_gpu, w, cap, [7, 11, 13, 17], rng)
    assert sh == sg
    if sh == 0:
        for a, c in zip(h, gp):
            assert np.array_equal(np.asarray(a), np.asarray(c))


def test_dmc_generations_on_the_host_split_join(monkeypatch):
    from test_gpu_dmc import test_dmc_generations_match_oracle
    monkeypatch.setenv("QMCW_HOST_SPLIT_JOIN", "1")
    test_dmc_generations_match_oracle("c2_dimer", 0.3, 1)
