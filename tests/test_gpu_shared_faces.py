"""Fluxes and EMFs of a stage that computes the ghost faces along x1 and x2 once (the
default launch of a uniform grid) against the four separate launches, in which every
block computes its own: HAMR_F1-F3 over all faces of a block and the transverse ghost
layer (those beyond two sides among them), HAMR_EMF and HAMR_ECENT, bit for bit, with
the arrays overwritten before either.  Two steps of each give the same state and
Courant dt.  Grids: the torus, and periodic boxes whose blocks meet on both sides of
x1 or x2, or meet themselves."""
import numpy as np
import pytest

pytest.importorskip("torch")

import hamr_gamma_wind_amd as H

pytestmark = pytest.mark.gpu

NG = 3
STALE = -7.25
ARRAYS = (H.HAMR_F1, H.HAMR_F2, H.HAMR_F3, H.HAMR_EMF, H.HAMR_ECENT)
TORUS = ((9, 11, 13), (3, 2, 2), 0)
BOXES = [((6, 8, 7), (2, 3, 2), 1), ((7, 6, 9), (3, 2, 1), 1), ((8, 6, 6), (1, 2, 1), 1), ((6, 7, 10), (1, 1, 1), 1)]


def _state(ctx, bs):
    """Random interior states with subluminal velocities and unequal mass fluxes."""
    rng = np.random.default_rng(5 + sum(bs))
    p, ps = np.zeros((ctx.nblk, 9) + ctx.D), np.zeros((ctx.nblk, 3) + ctx.D)
    I = (Ellipsis,) + (slice(NG, -NG),) * 3
    p[I] = rng.uniform(0.5, 1.0, (ctx.nblk, 9) + bs)
    p[(slice(None), slice(2, 8)) + I[1:]] = 0.1 * rng.normal(size=(ctx.nblk, 6) + bs)
    ps[I] = 0.1 * rng.normal(size=(ctx.nblk, 3) + bs)
    return p, ps


def _written(which, bs):
    """The cells of array `which` that a stage writes."""
    if which == H.HAMR_EMF:
        return tuple(slice(NG, NG + n + 1) for n in bs)
    d = which - H.HAMR_F1
    return tuple(slice(NG if k == d else NG - 1, NG + n + 1) for k, n in enumerate(bs))


@pytest.mark.parametrize("mode", ["fp64", "mixed", "hllc", "hllc mixed"])
@pytest.mark.parametrize("bs,nb,minkowski", [TORUS] + BOXES)
def test_every_flux_and_emf(bs, nb, minkowski, mode):
    ctx = H.Context(H.make_desc(bs, nb, minkowski=minkowski))
    try:
        ctx.set_grid()
        if minkowski:
            p, ps = _state(ctx, bs)
        else:
            ctx.init_torus(H.torus_desc())
            p, ps = ctx.get(H.HAMR_P), ctx.get(H.HAMR_PS)
        ctx.set_precision(H.HAMR_PREC_MIXED if "mixed" in mode else H.HAMR_PREC_FP64)
        if "hllc" in mode:
            ctx.set_riemann(H.HAMR_RIEMANN_HLLC)
        slot = H.HAMR_TUNE_NAMES.index("emf_centre")
        tile = ctx.tune_table()["flux1"]["threads"]
        out = []
        for threads in (tile, 64 if tile != 64 else 128):  # one size: one launch; two: four launches
            ctx.tune_set(slot, threads, 0, 1)
            ctx.set(H.HAMR_P, p)
            ctx.set(H.HAMR_PS, ps)
            for a in ARRAYS:
                ctx.set(a, np.full((ctx.nblk, H.NCOMP[a]) + ctx.D, STALE))
            ctx.stage_forward(1e-3)
            stage = [ctx.get(a) for a in ARRAYS]
            ctx.set(H.HAMR_P, p)
            ctx.set(H.HAMR_PS, ps)
            ctx.boundprim(1)
            dt = ctx.step(2, ctx.estimate_dt())
            out.append((stage, dt, ctx.get(H.HAMR_P), ctx.get(H.HAMR_PS), [ctx.get(a) for a in ARRAYS]))
    finally:
        ctx.close()
    one, four = out
    for a, x, y in zip(ARRAYS, one[0], four[0]):
        w = (Ellipsis,) + _written(a, bs)
        assert np.isfinite(y[w]).all() and not (y[w] == STALE).any()
        assert np.array_equal(x, y), a  # and nothing else is touched
    assert one[1] == four[1] and np.array_equal(one[2], four[2]) and np.array_equal(one[3], four[3])
    for a, x, y in zip(ARRAYS, one[4], four[4]):
        assert np.array_equal(x, y), a
