"""The adjoint's x1 and x2 reconstruction in segments of 8, 16 and 32 cells with a
shorter last one, against segments of 4: a box of a state repeated twice along each
direction, with the step halved as the spacing is, has the gradient of the single box
repeated, and every sum of both has the same terms in the same order, so that they are
equal bit for bit.  (Segments of 4 are checked against a reference gradient by the
boxes of test_gpu_adjoint_sizes.py.)"""
import numpy as np
import pytest

import hamr_gamma_wind_amd as H
from hamr_gamma_wind_amd import workloads as W

pytestmark = pytest.mark.gpu

GAM = 13.0 / 9.0
NG = 3
I = (Ellipsis,) + (slice(NG, -NG),) * 3


def _segment(n):
    """launch_adjoint's rule: the longest that still makes four wavefronts a SIMD."""
    seg = 32
    while seg > 4 and 7 * int(np.prod(n)) // seg < 256 * 16 * 64:
        seg //= 2
    return seg


def _gradient(prims, faces, w, rate):
    n = prims.shape[1:]
    desc = H.make_desc(n, (1, 1, 1), gam=GAM, minkowski=1, rho_floor=0.0, u_floor=0.0)
    ctx = H.Context(desc)
    try:
        ctx.set_grid()
        p, ps = W.to_block(prims, faces)
        ctx.set(H.HAMR_P, p)
        ctx.set(H.HAMR_PS, ps)
        weights = np.zeros(p.shape)
        weights[I] = w
        dx = H.desc_coords(desc)[1]
        gp, gps = ctx.stage_adjoint(rate * dx[0], weights)
        return gp[I][0], gps[I][0], dx
    finally:
        ctx.close()


@pytest.mark.parametrize("n,seg", [((33, 35, 35), 8), ((43, 45, 41), 16), ((55, 53, 53), 32)])
def test_repeated_box(n, seg):
    big = tuple(2 * k for k in n)
    assert _segment(n) == 4 and _segment(big) == seg and big[0] % seg and big[1] % seg
    prims, faces = W.minkowski_box(n, gam=GAM, seed=41)
    w = np.random.default_rng(42).normal(size=(9,) + n)
    rep = (1, 2, 2, 2)
    one = _gradient(prims, faces, w, 0.3)
    two = _gradient(np.tile(prims, rep), np.tile(faces, rep), np.tile(w, rep), 0.3)
    assert all(a == 2 * b for a, b in zip(one[2], two[2]))
    for a, b in zip(one, two[:2]):
        assert np.abs(a).max() > 0.0 and np.array_equal(np.tile(a, rep), b)
