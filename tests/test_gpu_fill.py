"""The one-launch ghost fill of a uniform grid against the oracle's three stages,
bit for bit, on block shapes and counts at its edges: the smallest block, one
block around the axis (its own pole partner), two, odd extents, a periodic box,
radial inflow that the outflow rule has to stop.

Every primitive, flag and face-field component of every ghost must equal the cell of
the oracle's global grid, except the face-field components that no stage fills
(B^1 beyond a radial edge, B^2 beyond the axis), which must be left as they were.
"""
import numpy as np
import pytest

import hamr_gamma_wind_amd as H
from tests import gridtools as GT

pytestmark = pytest.mark.gpu

NG = 3


@pytest.mark.parametrize("bs,nb,minkowski", [
    ((6, 6, 6), (1, 1, 1), 0),
    ((6, 6, 6), (2, 1, 2), 0),
    ((7, 9, 8), (2, 1, 1), 0),
    ((10, 13, 9), (3, 2, 2), 0),
    ((6, 7, 11), (1, 3, 4), 0),
    ((9, 6, 7), (1, 1, 1), 1),
    ((6, 8, 7), (2, 3, 2), 1),
])
def test_fill_equals_the_three_stages(oracle, bs, nb, minkowski):
    desc = H.make_desc(bs, nb, minkowski=minkowski)
    ctx = H.Context(desc)
    ctx.set_grid()
    rng = np.random.default_rng(sum(bs) + 7 * sum(nb))
    p = np.zeros((ctx.nblk, 9) + ctx.D)
    ps = np.full((ctx.nblk, 3) + ctx.D, np.nan)  # what no stage fills stays NaN
    I = (slice(NG, -NG),) * 3
    p[(slice(None), slice(None)) + I] = rng.uniform(0.1, 1.0, (ctx.nblk, 9) + bs)
    p[(slice(None), slice(2, 5)) + I] *= rng.choice([-0.2, 0.2], (ctx.nblk, 3) + bs)  # in- and outflow
    ps[(slice(None), slice(None)) + I] = rng.normal(size=(ctx.nblk, 3) + bs)
    ctx.set(H.HAMR_P, p)
    ctx.set(H.HAMR_PS, ps)
    ctx.boundprim(1)
    got_p, got_s = ctx.get(H.HAMR_P), ctx.get(H.HAMR_PS)
    ctx.close()
    grid = GT.oracle_grid(oracle, desc)
    P, S = GT.blocks_to_global(desc, p), GT.blocks_to_global(desc, ps)
    G = np.full_like(S, np.nan)
    G[:, NG:-NG, NG:-NG, NG:-NG] = S[:, NG:-NG, NG:-NG, NG:-NG]
    grid.bound(P, G)
    want_p, want_s = GT.global_to_blocks(desc, P), GT.global_to_blocks(desc, G)
    assert np.array_equal(got_p, want_p)
    # a block's own copy of an upper face is the neighbour's lower face on the
    # global grid; beyond the last block it is not filled on either side
    assert np.array_equal(np.isnan(got_s), np.isnan(want_s))
    assert np.array_equal(np.nan_to_num(got_s), np.nan_to_num(want_s))
