"""torch.autograd.Function over one forward stage of the step and its
hand-written adjoint (libhamr_hip.so).

torch holds the device memory; the library computes on its own stream.  The
forward copies the primitives and face fields from the given device tensors
into the context, runs the stage and returns U' (interior cells; ghost cells
are zero).  The backward runs the adjoint for the incoming gradient of U', which
the library reads in place, and returns dL/dP and dL/d(face field).  Both
synchronise torch's current stream before the library reads torch memory, and the
library's stream has finished when they return.
"""
import torch

from . import HamrError


class Stage(torch.autograd.Function):
    """U' = stage(P, face field) for a flat periodic box of one block (FP64)."""

    @staticmethod
    def forward(ctx, P, PS, hctx, Dt):
        for t, nc in ((P, 9), (PS, 3)):
            if t.dtype != torch.float64 or not t.is_cuda or not t.is_contiguous():
                raise HamrError("Stage: P and PS must be contiguous float64 device tensors")
            if tuple(t.shape) != (hctx.nblk, nc) + tuple(hctx.D):
                raise HamrError("Stage: tensor shape does not match the context layout")
        torch.cuda.current_stream().synchronize()
        U = torch.empty_like(P)
        hctx.stage_forward_dev(Dt, P.data_ptr(), PS.data_ptr(), U.data_ptr())
        ctx.hctx = hctx
        ctx.Dt = Dt
        ctx.save_for_backward(P, PS)
        return U

    @staticmethod
    def backward(ctx, gU):
        P, PS = ctx.saved_tensors
        hctx = ctx.hctx
        # the values themselves (a lazily negated view keeps its sign in a flag); the
        # weights of ghost cells are not read
        w = gU.resolve_neg().contiguous()
        gP = torch.empty_like(P)
        gPS = torch.empty_like(PS)
        torch.cuda.current_stream().synchronize()
        hctx.stage_grad_dev(ctx.Dt, P.data_ptr(), PS.data_ptr(), w.data_ptr(), gP.data_ptr(), gPS.data_ptr())
        return gP, gPS, None, None


def stage(P, PS, hctx, Dt):
    return Stage.apply(P, PS, hctx, Dt)
