"""The in-place wall pass with one thread per ordinate of a speed ring: ring
sizes that do and do not divide the block, the longest ring it takes (256),
one it leaves to the ordered walk (300), blocks that are not full, and
elements with two wall sides (the square's corners).  Against the FP64 CPU
oracle's ordered sweep: 1e-10 in FP64 (the same operations), 1e-5 in FP32."""
import numpy as np
import pytest

from small_cases import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tol", [(0, 1e-10), (1, 1e-5)])
@pytest.mark.parametrize("rorder,torder", [(5, 9), (8, 16), (3, 70), (2, 256), (1, 300)])
def test_ring_rounds_match_the_ordered_sweep(rorder, torder, precision, tol):
    from dgbgk import cases, meshgen
    from dgbgk.solver import Solver
    from oracle_py import OracleRun
    m = meshgen.unit_square(3, left=3, right=4, bottom=4, top=3, tw=1, alpha100=50)
    eta, w = cases.gauss_legendre_speeds(rorder)
    case = cases.Case("closed_box", m, eta, w, torder,
                      cases.base_params(u0=0.3, kn=0.2, length=1.0, rv=5.0, alpha=0.4))
    print(f"case closed box {rorder}x{torder} precision={precision}", flush=True)
    s, o = Solver(case, precision=precision), OracleRun(case)
    rs, ro = s.step(4), o.step(4)
    assert rel_l2(s.get_f(), o.get_f()) < tol
    assert np.allclose([r["sumres"] for r in rs], [r["sumres"] for r in ro], rtol=100 * tol)
