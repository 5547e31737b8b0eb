"""The sweeps' workgroup at the edges of its split: grids whose strips have
few blocks of 8 steps (fewer than its loaders run ahead), a last strip of one
row, one row more than a strip, and widths around the 16-column rounding. Two
whole steps against the oracle, bit for bit (sequential dot order).

And the fused vector update where vector operations take every cell (level
3): the same iterates as the separate kernels, bit for bit, alone and in a
batch, also where the budget ends after an odd and an even iteration (the
last s then lies in either array)."""
import os

import numpy as np
import pytest

import oracle_lib as ol
from gpu_util import compare_fields

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level,w,h", [(3, 17, 65), (4, 64, 64), (5, 33, 129), (6, 49, 65), (7, 65, 63), (7, 193, 66)])
def test_small_strips_match_oracle(level, w, h):
    import ifl_fluids as F
    sc = ol.REF_SCENES[level]
    print(f"level {level} {w}x{h}", flush=True)
    orc = ol.OracleSolver(level, w, h, sc["params"], sc["bodies"], fresh=True)
    bodies = [F.SolidBox(*b[1:]) if b[0] == F.BODY_BOX else F.SolidSphere(b[1], b[2], b[3], *b[5:]) for b in sc["bodies"]]
    gpu = F.FluidSolver(level, w, h, sc["params"], bodies, dot_order=F.DOT_SEQUENTIAL)
    for _ in range(2):
        orc.add_inflow(*sc["inflow"])
        gpu.add_inflow(*sc["inflow"])
        orc.update(sc["dt"])
        gpu.update(sc["dt"])
    for f in ol.state_fields(level):
        a, b = orc.field(f), gpu.field(f)
        if a is not None or b is not None:
            assert a.tobytes() == b.tobytes(), f"field {f}"
    gpu.close()
    orc.close()


def _solvers(level, sizes, fused, limit):
    import ifl_fluids as F
    sc = ol.REF_SCENES[level]
    bodies = [F.SolidBox(*b[1:]) if b[0] == F.BODY_BOX else F.SolidSphere(b[1], b[2], b[3], *b[5:]) for b in sc["bodies"]]
    old = os.environ.get("IFL_NO_FUSED_UPDATE")
    os.environ["IFL_NO_FUSED_UPDATE"] = "0" if fused else "1"
    try:
        kw = {} if limit is None else {"pcg_limit": limit}
        return [F.FluidSolver(level, w, h, sc["params"], bodies, dot_order=F.DOT_TREE, **kw) for w, h in sizes]
    finally:
        if old is None:
            del os.environ["IFL_NO_FUSED_UPDATE"]
        else:
            os.environ["IFL_NO_FUSED_UPDATE"] = old


@pytest.mark.parametrize("batch", [False, True])
@pytest.mark.parametrize("level,limit", [(3, None), (3, 7), (3, 8)])
def test_fused_update_every_cell(level, limit, batch):
    import ifl_fluids as F
    sc = ol.REF_SCENES[level]
    sizes = [(96, 80), (130, 67)] if batch else [(130, 67)]
    out = []
    for fused in (True, False):
        print(f"level {level} limit {limit} batch {batch} fused {fused}", flush=True)
        ss = _solvers(level, sizes, fused, limit)
        group = F.Batch(ss) if batch else None
        for _ in range(2):
            for s in ss:
                s.add_inflow(*sc["inflow"])
            if batch:
                group.update(sc["dt"])
            else:
                ss[0].update(sc["dt"])
        if batch:
            group.close()
        out.append(ss)
    for a, b in zip(*out):
        bad = compare_fields(a, b, ol.state_fields(level), where=f"level {level}")
        assert not bad, "\n".join(bad[:6])
        assert np.isfinite(a.field(F.Q_D * 16 + F.QF_SRC)).all()
        a.close()
        b.close()
