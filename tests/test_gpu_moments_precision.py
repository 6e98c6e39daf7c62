"""The FP32-bulk form's moment sums are FP64 and compensated in every moments
kernel.  Against long double sums of the same f: the density is within the
rounding of its own result (a uniform error of half an ulp is 0.29 ulp RMS,
6.4e-17 relative at the least and 1.3e-16 at the most over a binade; 7.4e-17 on
these states), where plain FP64 sums of 32 ordinates a wavefront are at 1.5e-16;
bounds 1e-16 RMS for n, twice that for u and p, and for v 1e-16 of the thermal
speed (1)."""
import numpy as np
import pytest

from small_cases import cylinder_small

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("split", [None, "1", "4"])
@pytest.mark.parametrize("rorder,torder", [(8, 16), (8, 32), (7, 19), (16, 32)])
def test_fp32_sums_are_compensated(rorder, torder, split, monkeypatch):
    from dgbgk import _lib
    from dgbgk.solver import Solver
    if split:
        monkeypatch.setenv("DGBGK_MOM_SPLIT", split)
    case = cylinder_small(elems=1200, rorder=rorder, torder=torder)
    print(f"case moment sums {rorder}x{torder} split={split}", flush=True)
    s = Solver(case, precision=_lib.DGBGK_FP32)
    s.step(3)
    f = s.get_f() * (1 + 0.3 * np.random.default_rng(2).random((s.E, s.V, 3)))
    f = f.astype(np.float32).astype(np.float64)
    s.set_f(f)
    nf, t, rv, pi = s.node_fields(), s.tables(), case.prm["rv"], 3.1416
    eta, th = t["vcord"][:, 0], t["vcord"][:, 1] * pi
    w = t["vcord"][:, 2] * (pi * rv * rv * 0.25 * (eta + 1)) * (4.0 / t["sumweight"])
    L = np.longdouble
    w, cx, cy = (a.astype(L) for a in (w, rv / 2 * (eta + 1) * np.cos(th),
                                       rv / 2 * (eta + 1) * np.sin(th)))
    def total(x):
        return (f.astype(L) * x[None, :, None]).sum(axis=1)
    n = total(w)
    u, v = total(w * cx) / n, total(w * cy) / n
    p = total(w * (cx * cx + cy * cy) / 2) - n * (u * u + v * v) / 2
    p *= L(case.prm["m"]) / L(6.022e26)
    def rms(x):
        return float(np.sqrt((x * x).mean()))
    assert rms(nf["disnd"] / n - 1) < 1e-16
    assert rms(nf["disux"] - u) < 2e-16 * rms(u)
    assert rms(nf["disuy"] - v) < 1e-16
    assert rms(nf["disps"] / p - 1) < 2e-16


@pytest.mark.parametrize("elems,rorder,torder", [(1200, 16, 32), (8000, 8, 16), (8000, 16, 32),
                                                 (12000, 8, 32)])
def test_fp64_density_is_no_further_off_than_the_other_kernels(elems, rorder, torder):
    """FP64 sums are plain; the density of the kernel that holds a node's
    ordinates within k_moments' own error, 1.2-1.45e-16 RMS of the exact sum
    at these sizes (a wavefront's 32 ordinates in one chain and its shares in
    another: 1.7-2.0e-16)."""
    from dgbgk.solver import Solver
    case = cylinder_small(elems=elems, rorder=rorder, torder=torder)
    print(f"case FP64 density {elems} {rorder}x{torder}", flush=True)
    s = Solver(case)
    s.step(3)
    f = s.get_f() * (1 + 0.3 * np.random.default_rng(2).random((s.E, s.V, 3)))
    s.set_f(f)
    t, rv, pi = s.tables(), case.prm["rv"], 3.1416
    w = t["vcord"][:, 2] * (pi * rv * rv * 0.25 * (t["vcord"][:, 0] + 1)) * (4.0 / t["sumweight"])
    n = np.zeros((s.E, 3), np.longdouble)
    for v in range(s.V):
        n += f[:, v].astype(np.longdouble) * np.longdouble(w[v])
    err = s.node_fields()["disnd"] / n - 1
    assert float(np.sqrt((err * err).mean())) < 1.4e-16
