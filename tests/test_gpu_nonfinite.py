"""Non-finite values travel as in the reference.  A side whose normal an
ordinate is parallel to takes the right element's values, so NaN or infinity
crosses it from right to left only: after a step from a state with a few
non-finite values, the same values are non-finite as in the FP64 CPU oracle
(FP64), or a subset of them (FP32, whose differences of nearby values meet
fewer)."""
import numpy as np
import pytest

from small_cases import c1, cylinder_small, lobatto10_walls

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("make", [c1, cylinder_small, lobatto10_walls])
def test_non_finite_values_spread_as_the_reference(make, bad, precision):
    from dgbgk.solver import Solver
    from oracle_py import OracleRun
    case = make()
    print(f"case non-finite {case.name} {bad} precision={precision}", flush=True)
    s, o = Solver(case, precision=precision), OracleRun(case)
    f = o.get_f().copy()
    rng = np.random.default_rng(5)
    for e in rng.choice(s.E, 12, replace=False):
        f[e, rng.integers(s.V), rng.integers(3)] = bad
    for e in rng.choice(s.E, 6, replace=False):  # at every ordinate
        f[e, :, rng.integers(3)] = bad
    s.set_f(f)
    o.set_f(f)
    s.step(1)
    o.step(1)
    got, want = ~np.isfinite(s.get_f()), ~np.isfinite(o.get_f())
    assert not (got & ~want).any()
    assert precision == 1 or np.array_equal(got, want)
