"""Results on their way to the caller: arrays that come through pinned memory
(up to 524,288 doubles a call) and larger ones copied straight, at the sizes
on either side, into arrays that hold other values before, and calls that ask
for some of the arrays only.  The same walkers in a small engine give the same
bits."""
import ctypes as C

import numpy as np
import pytest

from champ_amd import system
from champ_amd.engine import Engine

pytestmark = pytest.mark.gpu

KEYS = ("logpsid", "sign", "psij", "grad", "divv", "eloc", "epot")


def _engine(s, x):
    e = Engine(s, len(x))
    e.set_group_width(8)
    e.set_walkers(x)
    return e


@pytest.mark.parametrize("W", [16383, 16384, 16385])
@pytest.mark.parametrize("want", [KEYS, ("grad",), ("divv", "eloc"), ("logpsid",)], ids="-".join)
def test_full_evaluation(W, want):
    s = system.c2_dimer(2)
    x = system.random_walkers(s, W, seed=4)
    e = _engine(s, x)
    shape = {"grad": (W, s.nelec, 3), "divv": (W, s.nelec)}
    out = {k: np.full(shape.get(k, (W,)), np.nan) for k in want}
    p = lambda k: out[k].ctypes.data_as(C.POINTER(C.c_double)) if k in out else None
    assert e.lib.qmcw_eval_full(e.h, *[p(k) for k in KEYS]) == 0
    e.close()
    for part in (slice(0, 24), slice(W - 25, W)):
        e = _engine(s, x[part])
        ref = e.psi_at()
        e.close()
        for k in want:
            assert np.array_equal(out[k][part], ref[k]), k


@pytest.mark.parametrize("W", [1083, 1084])
@pytest.mark.parametrize("want", [(1, 1), (1, 0), (0, 1)])
def test_derivatives(W, want):
    s = system.c2_dimer(2, derivs=True)
    x = system.random_walkers(s, W, seed=4)
    e = _engine(s, x)
    out = [np.full((W, e.P), np.nan) if q else None for q in want]
    assert e.P == 242
    p = lambda a: None if a is None else a.ctypes.data_as(C.POINTER(C.c_double))
    assert e.lib.qmcw_derivs(e.h, p(out[0]), p(out[1])) == 0
    e.close()
    for part in (slice(0, 24), slice(W - 25, W)):
        e = _engine(s, x[part])
        ref = e.derivs()
        e.close()
        for a, r in zip(out, ref):
            assert a is None or np.array_equal(a[part], r)
