"""Small meshes' steps leave their epilogue to the next step's update, and a
batch ends with its own: the same steps in batches of other lengths (graphs,
their remainders, single steps, across the 1000th step's point gather) give
the same f and records to the last bit, with both block sizes and with one and
four lanes per node in the moments."""
import numpy as np
import pytest

from small_cases import cylinder_small

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("elems,rorder,torder,precision,slots", [
    (600, 6, 7, 0, 256), (600, 8, 16, 1, 256), (600, 8, 32, 0, 512), (9000, 2, 8, 0, 256),
    (7500, 8, 16, 0, 256)])
def test_batches_agree(elems, rorder, torder, precision, slots, monkeypatch):
    from dgbgk.solver import Solver
    monkeypatch.setenv("DGBGK_SLOTS", str(slots))
    case = cylinder_small(elems=elems, rorder=rorder, torder=torder)
    print(f"case batches {elems} {rorder}x{torder} precision={precision} slots={slots}", flush=True)
    a, b = Solver(case, precision=precision), Solver(case, precision=precision)
    ra = list(a.step(1003))
    rb = []
    for n in (1, 1, 2, 130, 860, 5, 1, 3):
        rb += list(b.step(n))
    assert len(ra) == len(rb) == 1003
    for i, (x, y) in enumerate(zip(ra, rb)):
        for k in ("sumres", "dte", "mass", "lift", "drag", "change"):
            assert x[k] == y[k], (i, k)
    assert ra[0]["drag"] == ra[998]["drag"] != ra[999]["drag"]  # the gather
    assert np.array_equal(a.get_f(), b.get_f(), equal_nan=True)
