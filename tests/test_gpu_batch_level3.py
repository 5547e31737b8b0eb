"""A level 3 batch folds the vector update into the product up to 2M cells and
keeps the two kernels above (levels 6-8 always fold): on both sides of the
line, the same statistics and state as the same solvers stepped alone, bit for
bit, out of budget after an odd and an even iteration (the last directions
then lie in either of a folding solver's two arrays)."""
import pytest

import oracle_lib as ol
from gpu_util import compare_fields, make_product

pytestmark = pytest.mark.gpu

UNDER = [(1024, 976), (1024, 976)]  # 1,998,848 cells
OVER = [(1024, 976), (1025, 977)]   # 2,000,849 cells


@pytest.mark.parametrize("limit", [7, 8])
@pytest.mark.parametrize("sizes", [UNDER, OVER], ids=["under", "over"])
def test_level3_batch_matches_solvers_alone(sizes, limit):
    import ifl_fluids as F
    sc = ol.REF_SCENES[3]
    make = lambda: [make_product(3, w, h, sc["params"], [], pcg_limit=limit) for w, h in sizes]
    print(f"level 3 batch {sizes} limit {limit}", flush=True)
    alone, together = make(), make()
    batch = F.Batch(together)
    for s in alone + together:
        s.add_inflow(*sc["inflow"])
    ra = [s.update(sc["dt"]).pressure for s in alone]
    rb = [st.pressure for st in batch.update(sc["dt"])]
    assert [(x.status, x.iterations, x.max_error) for x in ra] == [(x.status, x.iterations, x.max_error) for x in rb]
    assert all(x.status == F.SOLVE_BUDGET for x in ra)
    batch.close()
    for a, b in zip(alone, together):
        bad = compare_fields(a, b, ol.state_fields(3), where=f"{a.w}x{a.h}")
        assert not bad, "\n".join(bad[:6])
        a.close()
        b.close()
