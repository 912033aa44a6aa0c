"""The merged launch of fluxes and centre EMFs where its shape changes: after the tuner
has chosen the shapes of a uniform grid, and, in FP32, on a grid whose classes are
taken chunk by chunk with a remainder (from four chunks of 2^20 threads per class on).
State and Courant dt of the steps stay the same bits."""
import numpy as np
import pytest

pytest.importorskip("torch")

import hamr_gamma_wind_amd as H

pytestmark = pytest.mark.gpu

SLOT = H.HAMR_TUNE_NAMES.index("emf_centre")


def _start(grid, mixed, hllc=False):
    ctx = H.Context(H.make_desc(*grid))
    ctx.set_grid()
    ctx.init_torus(H.torus_desc())
    ctx.set_precision(H.HAMR_PREC_MIXED if mixed else H.HAMR_PREC_FP64)
    if hllc:
        ctx.set_riemann(H.HAMR_RIEMANN_HLLC)
    ctx.boundprim(1)
    return ctx, ctx.get(H.HAMR_P), ctx.get(H.HAMR_PS)


def _steps(ctx, p, ps, n, graph=False):
    ctx.set(H.HAMR_P, p)
    ctx.set(H.HAMR_PS, ps)
    return ctx.step(n, ctx.estimate_dt(), graph=graph), ctx.get(H.HAMR_P), ctx.get(H.HAMR_PS)


def _same(a, b):
    return a[0] == b[0] and np.array_equal(a[1], b[1]) and np.array_equal(a[2], b[2])


@pytest.mark.parametrize("mode", ["fp64", "mixed", "hllc", "hllc mixed"])
def test_tuned_shapes(mode):
    ctx, p, ps = _start(((9, 11, 13), (3, 2, 2)), "mixed" in mode, "hllc" in mode)
    try:
        before = _steps(ctx, p, ps, 2)
        ctx.set(H.HAMR_P, p)
        ctx.set(H.HAMR_PS, ps)
        table = ctx.autotune(2)
        assert all(table[k]["ms"] > 0.0 for k in ("flux1", "flux2", "flux3", "emf_centre"))
        assert np.array_equal(ctx.get(H.HAMR_P), p) and np.array_equal(ctx.get(H.HAMR_PS), ps)
        for graph in (False, True):
            assert _same(_steps(ctx, p, ps, 2, graph), before)
    finally:
        ctx.close()


def test_chunks():
    bs, nb = (32, 32, 32), (8, 5, 4)
    ctx, p, ps = _start((bs, nb), True)
    try:
        threads = ctx.tune_table()["flux1"]["threads"]
        items = int(np.prod(nb)) * (32 * 32 * 33 // threads)  # the smallest class, without its ghost faces
        chunk = (1 << 20) // threads
        assert items > 5 * chunk and items % chunk
        one = _steps(ctx, p, ps, 1)
        ctx.tune_set(SLOT, 64 if threads != 64 else 128, 0, 1)  # four launches
        assert _same(_steps(ctx, p, ps, 1), one)
    finally:
        ctx.close()
