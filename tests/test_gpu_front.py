"""Fluxes and centre EMFs in one launch against the four launches one after the
other: the same step bit for bit, with the same Courant dt.  The single launch takes
the classes in turn, and for FP32 launches of 16384 items or more per class in chunks
of 4096 with a remainder (256x128x128 zones, 18 k items per class); each block's ghost
faces along x1 and x2 come from the blocks beside it, and are computed where there is
none (radial edges, the axis; one block around it, one block in all).  Slots of
different workgroup sizes do not merge."""
import numpy as np
import pytest

pytest.importorskip("torch")

import hamr_gamma_wind_amd as H
from hamr_gamma_wind_amd import workloads as W

pytestmark = pytest.mark.gpu

RAGGED = ((9, 11, 13), (3, 2, 2))
SINGLE = ((12, 10, 8), (1, 1, 1))
AROUND = ((6, 7, 14), (3, 3, 1))


@pytest.mark.parametrize("grid, mode", [(RAGGED, "fp64"), (RAGGED, "mixed"), (RAGGED, "hllc"), (RAGGED, "hllc mixed"),
                                        (SINGLE, "fp64"), (AROUND, "mixed"), (AROUND, "fp64"),
                                        (W.TORUS_256, "mixed")])
def test_one_launch_equals_four(grid, mode):
    ctx = H.Context(H.make_desc(*grid))
    try:
        ctx.set_grid()
        ctx.init_torus(H.torus_desc())
        ctx.set_precision(H.HAMR_PREC_MIXED if "mixed" in mode else H.HAMR_PREC_FP64)
        if "hllc" in mode:
            ctx.set_riemann(H.HAMR_RIEMANN_HLLC)
        ctx.boundprim(1)
        p, ps = ctx.get(H.HAMR_P), ctx.get(H.HAMR_PS)
        slot = H.HAMR_TUNE_NAMES.index("emf_centre")
        out = []
        for threads in (256, 128):
            ctx.tune_set(slot, threads, 0, 1)
            ctx.set(H.HAMR_P, p)
            ctx.set(H.HAMR_PS, ps)
            out.append((ctx.step(2, ctx.estimate_dt()), ctx.get(H.HAMR_P), ctx.get(H.HAMR_PS)))
        a, b = out
        assert a[0] == b[0] and np.array_equal(a[1], b[1]) and np.array_equal(a[2], b[2])
    finally:
        ctx.close()
