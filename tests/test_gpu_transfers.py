"""Transfers through pinned pieces: f of several pieces with a last one that
is not full, in both forms (FP32 takes two passes through the device's
scratch) and for a mesh in another element order.  Values are only moved, so
everything is exact."""
import numpy as np
import pytest

from small_cases import cylinder_small, shuffled

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("elems,rorder,torder", [(600, 2, 8), (2000, 8, 16), (2000, 20, 31)])
def test_f_round_trip(elems, rorder, torder, precision):
    from dgbgk.solver import Solver
    case, _ = shuffled(cylinder_small(elems=elems, rorder=rorder, torder=torder), 3)
    print(f"case f transfer {elems} {rorder}x{torder} precision={precision}", flush=True)
    s = Solver(case, precision=precision)
    f = np.random.default_rng(1).random((s.E, s.V, 3))
    f = f.astype(np.float32).astype(np.float64)
    s.set_f(f)
    assert np.array_equal(s.get_f(), f)
    s.step(1)
    g = s.get_f()
    assert np.array_equal(s.get_f(), g) and not np.array_equal(g, f)

