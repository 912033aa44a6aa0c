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
