"""Solves that end at every edge of the host loop's groups of iterations: out
of budget after 1, 4, 5, 8, 12, 13, 16, 17, 24, 25 and 28 iterations (the
first group, the first one ahead, the change of the group size, a group cut
short) and converged (no budget), on a small grid of one strip and on grids of
several, where the loop's rules differ. The same solver as a batch of one runs
the batch's own loop (groups doubling from 4), and one without the fused
vector update the separate kernels: statistics and the whole state have to be
the same, bit for bit, over two steps."""
import pytest

import oracle_lib as ol
from gpu_util import compare_fields, make_product

pytestmark = pytest.mark.gpu

BUDGETS = [1, 4, 5, 8, 12, 13, 16, 17, 24, 25, 28, None]


@pytest.mark.parametrize("level,w,h", [(3, 130, 67), (4, 48, 40), (5, 70, 130), (7, 48, 40), (7, 140, 130)])
def test_group_edges(level, w, h, monkeypatch):
    import ifl_fluids as F
    sc = ol.REF_SCENES[level]

    def run(budget, fused, batch):
        monkeypatch.setenv("IFL_NO_FUSED_UPDATE", "0" if fused else "1")
        kw = {} if budget is None else {"pcg_limit": budget}
        s = make_product(level, w, h, sc["params"], sc["bodies"], dot_order=F.DOT_TREE, **kw)
        group = F.Batch([s]) if batch else None
        rows = []
        for _ in range(2):
            s.add_inflow(*sc["inflow"])
            st = group.update(sc["dt"])[0] if batch else s.update(sc["dt"])
            rows += [(x.status, x.iterations, x.max_error) for x in (st.heat, st.pressure)]
        if batch:
            group.close()
        return s, rows

    for budget in BUDGETS:
        print(f"level {level} {w}x{h} budget {budget}", flush=True)
        a, ra = run(budget, True, False)
        assert all(r[0] == (F.SOLVE_CONVERGED if budget is None else F.SOLVE_BUDGET) for r in ra[1::2]), ra
        for fused, batch in ((True, True), (False, False)):
            b, rb = run(budget, fused, batch)
            where = f"level {level} {w}x{h} budget {budget} fused {fused} batch {batch}"
            assert ra == rb, where
            bad = compare_fields(a, b, ol.state_fields(level), where=where)
            assert not bad, "\n".join(bad[:6])
            b.close()
        a.close()
