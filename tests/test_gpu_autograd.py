"""The incoming gradient of torch.autograd in the forms the engine may hand it over in:
as it is, transposed, expanded, and as a lazily negated view (whose memory holds the
other sign) give the gradients of the same values, bit for bit."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import hamr_gamma_wind_amd as H
from hamr_gamma_wind_amd import workloads as W
from hamr_gamma_wind_amd.autograd import stage

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["transposed", "expanded", "negated", "negated and transposed"])
def test_forms_of_the_incoming_gradient(form):
    n = (9, 6, 11)
    ctx = H.Context(H.make_desc(n, (1, 1, 1), minkowski=1, rho_floor=0.0, u_floor=0.0))
    try:
        ctx.set_grid()
        p, ps = W.to_block(*W.minkowski_box(n, gam=13.0 / 9.0, seed=35))
        g = torch.tensor(np.random.default_rng(36).normal(size=p.shape), device="cuda:0")
        if form == "expanded":
            g = g[..., :1].expand(g.shape).contiguous()
            same = g[..., :1].expand(g.shape)
        else:
            same = torch._neg_view(-g) if "negated" in form else g
            if "transposed" in form:
                base = same.transpose(-1, -3)
                same = (torch._neg_view(-base.resolve_neg().contiguous()) if "negated" in form
                        else base.contiguous()).transpose(-1, -3)
        assert torch.equal(same, g)
        got = []
        for gU in (g, same):
            P = torch.tensor(p, device="cuda:0", requires_grad=True)
            PS = torch.tensor(ps, device="cuda:0", requires_grad=True)
            stage(P, PS, ctx, 1e-3).backward(gU)
            got.append((P.grad, PS.grad))
        assert got[0][0].abs().max() > 0.0
        assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    finally:
        ctx.close()
