"""Adjoint of one stage at the sizes where its gathers can go wrong: the
smallest box the library takes, z-rows that share a block, fill it in part or
exceed it by one, odd
numbers of rows, and lines of 28, 29 and 57 cells (the x1 and x2 tiles).

Same workload and bar as the 12x10x8 box: dL/dP and dL/d(face field) equal the
FP64 reference gradient to 1e-9 of each component's largest magnitude; a second
call gives the same bits (nothing is accumulated in varying order)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import hamr_gamma_wind_amd as H
from hamr_gamma_wind_amd import workloads as W
from tests import adjoint_reference as R
from tests import gridtools as GT

pytestmark = pytest.mark.gpu

GAM = 13.0 / 9.0
NG = 3


@pytest.mark.parametrize("n", [(6, 7, 6), (7, 6, 60), (8, 28, 61), (29, 6, 17), (57, 7, 16), (6, 6, 257)])
def test_gradient_equals_reference(n):
    desc = H.make_desc(n, (1, 1, 1), gam=GAM, minkowski=1, rho_floor=0.0, u_floor=0.0)
    ctx = H.Context(desc)
    try:
        ctx.set_grid()
        prims, faces = W.minkowski_box(n, gam=GAM, seed=31)
        p, ps = W.to_block(prims, faces)
        _, dx = H.desc_coords(desc)
        Dt = 0.3 * min(dx)
        w = np.random.default_rng(32).normal(size=(1, 9) + tuple(k + 2 * NG for k in n))
        got = []
        for _ in range(2):
            ctx.set(H.HAMR_P, p)
            ctx.set(H.HAMR_PS, ps)
            got.append(ctx.stage_adjoint(Dt, w))
    finally:
        ctx.close()
    gp, gps = got[0]
    assert np.array_equal(gp, got[1][0]) and np.array_equal(gps, got[1][1])
    I = (slice(None),) + tuple(slice(NG, NG + k) for k in n)
    Pt, PSt = torch.tensor(prims, requires_grad=True), torch.tensor(faces, requires_grad=True)
    (R.stage(Pt, PSt, Dt, dx, GAM) * torch.tensor(w[0][I])).sum().backward()
    eP = GT.relerr_by_var(gp[0][I][None], Pt.grad.numpy()[None])
    eS = GT.relerr_by_var(gps[0][I][None], PSt.grad.numpy()[None])
    print(n, "dL/dP", np.array2string(eP, precision=2), "dL/dB", np.array2string(eS, precision=2), flush=True)
    assert np.all(eP[:8] <= 1e-9) and np.abs(gp[0][8]).max() == 0.0
    assert np.all(eS <= 1e-9)


def _dev(a):
    return torch.tensor(a, device="cuda:0")


def test_buffers_in_place_and_overlapping():
    """The gradients are written in place where nothing overlaps them, else through
    the work arrays: over the weights, without dL/d(face field), and apart."""
    n = (9, 6, 11)
    ctx = H.Context(H.make_desc(n, (1, 1, 1), gam=GAM, minkowski=1, rho_floor=0.0, u_floor=0.0))
    try:
        ctx.set_grid()
        p, ps = (_dev(a) for a in W.to_block(*W.minkowski_box(n, gam=GAM, seed=33)))
        w = _dev(np.random.default_rng(34).normal(size=tuple(p.shape)))
        w[..., :NG] = float("nan")  # weights of ghosts are not read
        gp, gps = torch.full_like(p, float("nan")), torch.full_like(ps, float("nan"))
        torch.cuda.synchronize()
        state = (1e-3, p.data_ptr(), ps.data_ptr())
        ctx.stage_grad_dev(*state, w.data_ptr(), gp.data_ptr(), gps.data_ptr())
        assert torch.isfinite(gp).all() and torch.isfinite(gps).all()
        only, over = torch.zeros_like(p), w.clone()
        torch.cuda.synchronize()
        ctx.stage_grad_dev(*state, w.data_ptr(), only.data_ptr(), None)
        ctx.stage_grad_dev(*state, over.data_ptr(), over.data_ptr(), gps.data_ptr())
        assert torch.equal(only, gp) and torch.equal(over, gp)
    finally:
        ctx.close()


def test_stage_from_device_arrays_equals_the_steps():
    """hamr_stage_forward_dev of several blocks: set, forward, get, ghosts zeroed."""
    ctx = H.Context(H.make_desc((9, 10, 7), (2, 2, 2)))
    try:
        ctx.set_grid()
        ctx.init_torus(H.torus_desc())
        p, ps = _dev(ctx.get(H.HAMR_P)), _dev(ctx.get(H.HAMR_PS))
        U, V = torch.full_like(p, float("nan")), torch.empty_like(p)
        torch.cuda.synchronize()
        ctx.stage_forward_dev(1e-3, p.data_ptr(), ps.data_ptr(), U.data_ptr())
        got = ctx.get(H.HAMR_P), ctx.get(H.HAMR_PSH)
        ctx.set_dev(H.HAMR_P, p.data_ptr())
        ctx.set_dev(H.HAMR_PS, ps.data_ptr())
        ctx.stage_forward(1e-3)
        ctx.get_dev(H.HAMR_UNEW, V.data_ptr())
        I = (Ellipsis,) + (slice(NG, -NG),) * 3
        assert torch.equal(U[I], V[I])
        U[I] = 0.0
        assert not U.any()
        assert np.array_equal(got[0], ctx.get(H.HAMR_P)) and np.array_equal(got[1], ctx.get(H.HAMR_PSH))
    finally:
        ctx.close()
