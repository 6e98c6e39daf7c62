"""Both moments kernels on the checks of each: k_moments with the update's sums
(DGBGK_MOM_SPLIT asks for it where a small mesh would take the kernel that
holds a node's ordinates) fused and not, at both prefetch depths and tile
sizes, in graphs and eagerly; and k_moments_once's FP64 form of one lane per
node, which takes more than 320 blocks of 64 nodes, against the FP64 CPU
oracle.  Same operations: bit-identical; oracle: 1e-10 (another order of the
same FP64 sums)."""
import numpy as np
import pytest

from small_cases import cylinder_small, rel_l2

pytestmark = pytest.mark.gpu

FIELDS = ("disnd", "disux", "disuy", "disps", "mu")


def _epilogues(s, n):
    """Launches of the step's epilogue over n steps: every step with
    k_moments, one at the batch's end with k_moments_once."""
    s.timing(True)
    s.step(n)
    count = s.kernel_time(4)[1]
    s.timing(False)
    return count


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("split", ["1", "4", "8"])
def test_fused_sums_depth_and_slots_with_k_moments(split, precision, monkeypatch):
    from dgbgk.solver import Solver
    case = cylinder_small(elems=800, rorder=8, torder=16)
    print(f"case k_moments arms split={split} precision={precision}", flush=True)
    monkeypatch.setenv("DGBGK_MOM_SPLIT", split)
    runs = {}
    for fuse in ("1", "0"):
        for depth in ("1", "2"):
            for slots in ("256", "512"):
                monkeypatch.setenv("DGBGK_FUSE_MOMENTS", fuse)
                monkeypatch.setenv("DGBGK_PREFETCH", depth)
                monkeypatch.setenv("DGBGK_SLOTS", slots)
                s = Solver(case, precision=precision, vchunk=24)
                cfg = s.launch_config()
                assert (cfg["mom_split"], cfg["depth"], cfg["slots"]) == (
                    int(split), int(depth), int(slots))
                assert _epilogues(s, 3) == 3
                runs[fuse, depth, slots] = (s.get_f(), s.node_fields())
                s.close()
    f0, n0 = runs["1", "1", "256"]
    for arm, (f1, n1) in runs.items():
        assert np.array_equal(f1, f0), arm
        for k in FIELDS:
            assert np.array_equal(n1[k], n0[k]), (arm, k)


def test_fp32_default_depth_two_is_depth_one(monkeypatch):
    """The size from which FP32 keeps two ordinates in flight by itself."""
    from dgbgk.solver import Solver
    case = cylinder_small(elems=22000, rorder=13, torder=16)
    print("case FP32 depth two by size", flush=True)
    a = Solver(case, precision=1)
    assert a.launch_config()["depth"] == 2
    monkeypatch.setenv("DGBGK_PREFETCH", "1")
    b = Solver(case, precision=1, vchunk=a.launch_config()["vchunk"])
    assert b.launch_config()["depth"] == 1
    for fuse in (None, "4"):
        if fuse:
            monkeypatch.setenv("DGBGK_MOM_SPLIT", fuse)
            b.close()
            b = Solver(case, precision=1, vchunk=a.launch_config()["vchunk"])
            monkeypatch.setenv("DGBGK_PREFETCH", "2")
            a = Solver(case, precision=1, vchunk=a.launch_config()["vchunk"])
        assert a.step(3) == b.step(3)
        assert np.array_equal(a.get_f(), b.get_f())


@pytest.mark.parametrize("precision", [0, 1])
def test_graph_equals_eager_with_k_moments(precision, monkeypatch):
    from dgbgk.solver import Solver
    case = cylinder_small(elems=800)
    print(f"case graph vs eager, k_moments, precision={precision}", flush=True)
    monkeypatch.setenv("DGBGK_MOM_SPLIT", "4")
    a = Solver(case, precision=precision)
    monkeypatch.setenv("DGBGK_NO_GRAPH", "1")
    b = Solver(case, precision=precision)
    for n in (65, 64, 3, 128, 741, 2):  # across the 1000th step's point gather
        assert a.step(n) == b.step(n)
        assert np.array_equal(a.get_f(), b.get_f())
    assert a.itime == b.itime == 1003


@pytest.mark.parametrize("elems,rorder,torder,split", [
    (7500, 8, 16, 4), (7500, 6, 7, 4), (9000, 8, 32, 8), (7500, 7, 19, 8), (7500, 16, 32, 16),
    (7500, 3, 91, 16)])
def test_one_lane_per_node_matches_the_oracle(elems, rorder, torder, split):
    from dgbgk.solver import Solver
    from oracle_py import OracleRun
    case = cylinder_small(elems=elems, rorder=rorder, torder=torder)
    blocks = -(-3 * case.mesh.nelem // 64)
    print(f"case one lane per node {case.mesh.nelem} {rorder}x{torder}", flush=True)
    assert blocks > 320 and blocks * split <= 8192
    s, o = Solver(case), OracleRun(case)
    assert s.launch_config()["mom_split"] == split
    rs, ro = s.step(2), o.step(2)
    nf, no = s.node_fields(), o.node_fields()
    assert rel_l2(s.get_f(), o.get_f()) < 1e-10
    for k in ("disnd", "disps"):
        assert rel_l2(nf[k], no[k]) < 1e-10, k
    for a, b in zip(rs, ro):
        assert abs(a["mass"] - b["mass"]) < 1e-10 * b["mass"]
        assert abs(a["dte"] - b["dte"]) < 1e-10 * b["dte"]
    o.prepare_step()  # MU is COMPMU of the current f
    assert rel_l2(nf["mu"], o.node_fields()["mu"]) < 1e-10
    assert _epilogues(s, 3) == 1


@pytest.mark.parametrize("elems,rorder,torder,precision,slots", [
    (9000, 6, 9, 0, 256), (9000, 8, 16, 1, 512)])
def test_batches_of_many_blocks_agree(elems, rorder, torder, precision, slots, monkeypatch):
    """Stable flows (every value finite) of more than 320 blocks."""
    from dgbgk.solver import Solver
    monkeypatch.setenv("DGBGK_SLOTS", str(slots))
    case = cylinder_small(elems=elems, rorder=rorder, torder=torder)
    print(f"case batches {elems} {rorder}x{torder} precision={precision}", flush=True)
    a, b = Solver(case, precision=precision), Solver(case, precision=precision)
    ra = a.step(203)
    rb = [r for n in (1, 2, 66, 130, 1, 3) for r in b.step(n)]
    assert ra == rb
    f = a.get_f()
    assert np.isfinite(f).all() and np.array_equal(f, b.get_f())
