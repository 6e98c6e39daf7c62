"""Non-finite values travel as in the reference.  A side whose normal an
ordinate is parallel to takes the right element's values, so NaN or infinity
crosses it from right to left only: after a step from a state with a few
non-finite values, the same values are non-finite as in the FP64 CPU oracle
(FP64), or a subset of them (FP32, whose differences of nearby values meet
fewer).  And a seed of any state gives the Maxwellian formula's values: 0 where
its exponential underflows, NaN where the state is."""
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


@pytest.mark.parametrize("precision,tol", [(0, 1e-11), (1, 1e-6)])
@pytest.mark.parametrize("u,temp", [
    (0.1, 1.0), (30.0, 1.0), (1e30, 1.0), (np.inf, 1.0), (np.nan, 1.0), (0.1, 1e-3),
    (0.1, 1e-40), (0.1, 1e-300), (0.1, 0.0)])
def test_seed_of_extreme_states(u, temp, precision, tol):
    from dgbgk.solver import Solver
    # tolerance: the exponent's ten roundings at up to 745 (FP64), the store (FP32)
    case = c1(n=4)
    print(f"case seed u={u} T={temp} precision={precision}", flush=True)
    s = Solver(case, precision=precision)
    full = [np.full(case.mesh.npoin, x) for x in (1.0, u, 0.0, temp)]
    s.seed(*full)
    # src/inicon2.f90:149-163 with n = rho NA / M, beta^2 = rho / (2 rho R T)
    prm, vc = case.prm, s.tables()["vcord"]
    pr = prm["rgas"] * temp
    n = 6.022e26 / prm["m"] if pr > 0.0 else 0.0
    b2 = 1.0 / (2 * pr) if pr > 0.0 else 0.0
    th, rad = vc[:, 1] * 3.1416, (vc[:, 0] + 1) * prm["rv"] / 2
    with np.errstate(over="ignore", invalid="ignore", under="ignore"):
        want = n * (b2 / 3.1416) * np.exp(-b2 * ((rad * np.cos(th) - u) ** 2
                                                 + (rad * np.sin(th)) ** 2))
        want = want.astype(np.float32 if precision else np.float64).astype(np.float64)
    f = s.get_f()
    got = f[0, :, 0]
    assert np.array_equal(f, np.broadcast_to(got[None, :, None], f.shape), equal_nan=True)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and not np.isinf(got).any()
    ok = np.isfinite(want)
    assert np.all(np.abs(got[ok] - want[ok]) <= tol * np.abs(want[ok]) + 1e-30 * n * b2)
