"""The stages that hamr_time_stage times as a step launches them: fluxes with centre
EMFs, then corner EMFs, leave HAMR_F1-F3, HAMR_ECENT and HAMR_EMF as a stage does,
with the launches merged and apart; p and ps stay as they are."""
import numpy as np
import pytest

import hamr_gamma_wind_amd as H
from hamr_gamma_wind_amd import workloads as W

pytestmark = pytest.mark.gpu

ARRAYS = (H.HAMR_F1, H.HAMR_F2, H.HAMR_F3, H.HAMR_ECENT, H.HAMR_EMF)
FRONT, CORNER = 8, 9


@pytest.mark.parametrize("merged", [True, False])
@pytest.mark.parametrize("mixed", [False, True])
def test_fluxes_and_emfs(merged, mixed):
    n = (9, 7, 11)
    ctx = H.Context(H.make_desc(n, (1, 1, 1), minkowski=1))
    try:
        ctx.set_grid()
        ctx.set_precision(H.HAMR_PREC_MIXED if mixed else H.HAMR_PREC_FP64)
        if not merged:
            ctx.tune_set(H.HAMR_TUNE_NAMES.index("emf_centre"), 64, 0, 1)
        p, ps = W.to_block(*W.minkowski_box(n, seed=37))
        ctx.set(H.HAMR_P, p)
        ctx.set(H.HAMR_PS, ps)
        ctx.boundprim(1)
        p, ps = ctx.get(H.HAMR_P), ctx.get(H.HAMR_PS)
        for a in ARRAYS:
            ctx.set(a, np.full((1, H.NCOMP[a]) + ctx.D, -7.25))
        assert ctx.time_stage(FRONT, 2) > 0.0 and ctx.time_stage(CORNER, 2) > 0.0
        got = [ctx.get(a) for a in ARRAYS]
        assert np.array_equal(ctx.get(H.HAMR_P), p) and np.array_equal(ctx.get(H.HAMR_PS), ps)
        for a in ARRAYS:
            ctx.set(a, np.full((1, H.NCOMP[a]) + ctx.D, -7.25))
        ctx.stage_forward(1e-3)
        for a, g in zip(ARRAYS, got):
            assert (g != -7.25).any() and np.array_equal(g, ctx.get(a)), a
        with pytest.raises(H.HamrError):
            ctx.time_stage(CORNER + 1)
    finally:
        ctx.close()
