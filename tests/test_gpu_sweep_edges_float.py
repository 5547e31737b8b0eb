"""The single-precision sweeps at the edges of their workgroup's split: strips
of 10 blocks of 8 steps, fewer than their loaders run ahead (4 loaders of 3
blocks; in double precision the forward and backward loaders hold 8 and 6
blocks, and only the factor build's 12), the narrowest grid, last strips of one
and two rows. The forward sweep's loaders form and store the residual and take
max|r|: the statistics' max_error is max|r| of the residual that the solve
leaves, exactly, and that residual is b - A p of the p that it leaves, with A p
from the oracle's double-precision matrixVectorProduct. After at most 5
iterations each of the few operations on a cell's residual and p rounds once:
40 operations of 2^-53 of the largest magnitudes in play, doubled for the
deflated forms' shift by the mean, bound the difference."""
import numpy as np
import pytest

import oracle_lib as ol
from gpu_util import make_product

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level,w,h", [(3, 3, 65), (3, 17, 130), (5, 33, 65), (5, 49, 129), (7, 65, 63), (7, 70, 66)])
@pytest.mark.parametrize("form", ["mixed", "refine"])
def test_residual_and_its_maximum(form, level, w, h):
    import ifl_fluids as F
    sc = ol.REF_SCENES[level]
    orc = ol.OracleSolver(level, w, h, sc["params"], sc["bodies"], fresh=True)
    if level >= 4:
        for q in [ol.Q_D, ol.Q_U, ol.Q_V] + ([ol.Q_T] if level >= 6 else []):
            orc.stage("FILL_SOLID", q)
    if level >= 7:
        orc.stage("COMPUTE_DENSITIES")
    orc.stage("BUILD_PRESSURE", 0, sc["dt"])
    orc.stage("BUILD_PRECON")
    state = {f: orc.field(f) for f in ol.state_fields(level)}
    fluid = orc.field(ol.qfield(ol.Q_D, ol.QF_CELL)) == 0 if level >= 4 else np.ones(w * h, bool)
    norm = fluid if level >= 6 else np.ones(w * h, bool)  # the reference's norm domain
    # a seeded right-hand side over the FLUID cells (no inflow rectangle reaches a face of every such grid)
    b = np.where(fluid, np.random.default_rng(w + 1000 * h).uniform(-1.0, 1.0, w * h), 0.0)
    state[ol.F_R] = b
    adiag = np.abs(state[ol.F_ADIAG]).max()

    for limit in (1, 2, 5):
        gpu = make_product(level, w, h, sc["params"], sc["bodies"],
                           precision=F.PREC_MIXED if form == "mixed" else F.PREC_REFINE)
        gpu._push_bodies()
        for f, v in state.items():
            if v is not None:
                gpu.set_field(f, v)
        gpu.stage("BUILD_PRECON")
        st = F.SolveStats()
        gpu.stage("PROJECT", limit, stats=st)
        p, r = gpu.field(ol.F_P), gpu.field(ol.F_R)
        gpu.close()
        orc.set_field(ol.F_S, p)
        orc.stage("MATVEC")
        off = np.abs((b - orc.field(ol.F_Z)) - r)[fluid].max()
        bound = 80 * 2.0 ** -53 * limit * (4 * adiag * np.abs(p).max() + np.abs(b).max())
        print(f"{form} level {level} {w}x{h} limit {limit}: status {st.status}, max|r| {st.max_error:.3e}, "
              f"|b - A p - r| {off:.2e} (bound {bound:.2e}, max|b| {np.abs(b).max():.2e})", flush=True)
        assert np.isfinite(r).all() and st.status in (F.SOLVE_BUDGET, F.SOLVE_CONVERGED)
        assert st.max_error == np.abs(r[norm]).max()
        assert off <= bound
    orc.close()
