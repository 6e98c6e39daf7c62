"""The moments kernel that holds a node's ordinates in registers: shares of
4, 8 and 16 wavefronts, full, ragged and shorter than a run of four, a
wavefront without ordinates, the most it holds (512) and one more (513, the
other kernel's eight wavefronts per node).  Against the FP64 CPU oracle: 1e-10 in FP64 (the same sums in
another order), 1e-5 in FP32."""
import pytest

from small_cases import cylinder_small, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tol", [(0, 1e-10), (1, 1e-5)])
@pytest.mark.parametrize("rorder,torder,split", [
    (6, 7, 4), (8, 16, 4), (3, 43, 8), (8, 32, 8), (3, 90, 16), (16, 32, 16), (27, 19, 8)])
def test_one_read_moments(rorder, torder, split, precision, tol):
    from dgbgk.solver import Solver
    from oracle_py import OracleRun
    case = cylinder_small(elems=600, rorder=rorder, torder=torder)
    print(f"case moments {rorder}x{torder} precision={precision}", flush=True)
    s, o = Solver(case, precision=precision), OracleRun(case)
    assert s.launch_config()["mom_split"] == split
    rs, ro = s.step(3), o.step(3)
    assert rel_l2(s.get_f(), o.get_f()) < tol
    nf, no = s.node_fields(), o.node_fields()
    for k in ("disnd", "disps"):
        assert rel_l2(nf[k], no[k]) < tol, k
    for a, b in zip(rs, ro):
        assert abs(a["mass"] - b["mass"]) < tol * b["mass"]
        assert abs(a["dte"] - b["dte"]) < tol * b["dte"]
    # MU is COMPMU of the current f, the oracle's at the top of its next step
    o.prepare_step()
    assert rel_l2(nf["mu"], o.node_fields()["mu"]) < tol
