"""torch.autograd bindings of the EFF/OLA operator and of the TV prior.

    plan = OlaPlan(sx, sf, winaux)
    y    = ola(x, f, plan)                 # B(x, f), differentiable in x and f
    loss = 0.5 * ((y - obs) ** 2).sum() + lam * tv(x, eps)
    loss.backward()

The backward of ``ola`` is the exact adjoint pair (x-adjoint F'g and
f-adjoint X'g, olaGPU.py:261-311 without the patch-local truncation), run as
one fused launch sequence when both gradients are needed; it reuses the row
transforms of the forward when nothing else ran on the plan in between.
``tv`` is isotropic and eps-smoothed (the reference has no TV prior):
TV(x) = sum sqrt(dx^2 + dy^2 + eps^2), forward differences, zero past the
last row/column; its value and gradient are HIP kernels, and the gradient
reads the upstream scalar from device memory (no host synchronisation).
"""
import torch
import torch.autograd.forward_ad as fwAD

from . import _lib
from .optGPU import _Scratch


class _OlaFunction(torch.autograd.Function):

    @staticmethod
    def forward(ctx, x, f, plan, exact):
        y = plan.forward(x, f)
        ctx.plan = plan
        ctx.exact = bool(exact)
        ctx.save_for_backward(x, f)
        return y

    @staticmethod
    def backward(ctx, gy):
        x, f = ctx.saved_tensors
        plan = ctx.plan
        gy = gy.contiguous()
        need_x, need_f = ctx.needs_input_grad[0], ctx.needs_input_grad[1]
        gx = gf = None
        if need_x and need_f:
            gx, gf = plan.adjoint_xf(gy, x, f, exact=ctx.exact)
        elif need_x:
            gx = plan.adjoint_x(gy, f, exact=ctx.exact)
        elif need_f:
            gf = plan.adjoint_f(gy, x, exact=ctx.exact)
        return gx, gf, None, None


def ola(x, f, plan, exact=True):
    """Differentiable B(x, f) on `plan` (x: ([B,] H, W), f: ([B,] P, sf0, sf1))."""
    return _OlaFunction.apply(x, f, plan, exact)


class _TvFunction(torch.autograd.Function):

    @staticmethod
    def forward(ctx, x, eps):
        if x.dtype != torch.float32 or x.device.type != 'cuda':
            raise TypeError('tv: expected a float32 device tensor')
        xc = x.contiguous()
        H, W = int(xc.shape[-2]), int(xc.shape[-1])
        K = xc.numel() // (H * W)
        sc = _Scratch(xc.numel(), xc.device)
        val = torch.empty(1, dtype=torch.float64, device=xc.device)
        _lib.call('vmbd_tv', _lib.ptr(xc), K, H, W, float(eps), _lib.ptr(sc.partials), _lib.ptr(val),
                  _lib.stream_ptr())
        ctx.eps = float(eps)
        ctx.save_for_backward(xc)
        return val.to(torch.float32).reshape(())

    @staticmethod
    def backward(ctx, g):
        (x,) = ctx.saved_tensors
        H, W = int(x.shape[-2]), int(x.shape[-1])
        K = x.numel() // (H * W)
        scale = g.to(torch.float32).contiguous().reshape(1)
        out = torch.empty_like(x)
        _lib.call('vmbd_tv_grad', _lib.ptr(out), _lib.ptr(x), K, H, W, ctx.eps, _lib.ptr(scale), 1.0, 0,
                  _lib.stream_ptr())
        return out, None


def tv(x, eps=1e-3):
    """Isotropic eps-smoothed total variation, summed over all images of x."""
    return _TvFunction.apply(x, eps)


class _LossFunction(torch.autograd.Function):
    """1/2 |B(x, f) - y|^2 + lam TV(x) for a constant y: the residual is formed
    in the operator's final store and kept for the backward, which is linear in
    it; the upstream scalar is applied in the adjoints' final stores."""

    @staticmethod
    def forward(ctx, x, f, y, plan, lam, eps, exact):
        r = plan.forward(x, f, sub=y)
        xc = x.contiguous()
        H, W = int(xc.shape[-2]), int(xc.shape[-1])
        K = xc.numel() // (H * W)
        nb = _lib.lib().vmbd_reduce_blocks(max(r.numel(), xc.numel()))
        part = torch.empty(2 * nb, dtype=torch.float64, device=xc.device)
        val = torch.empty((), dtype=torch.float32, device=xc.device)
        _lib.call('vmbd_loss', _lib.ptr(r), r.numel(), _lib.ptr(xc), K, H, W, eps, lam, _lib.ptr(part), _lib.ptr(val),
                  _lib.stream_ptr())
        ctx.plan, ctx.lam, ctx.eps, ctx.exact = plan, lam, eps, exact
        ctx.save_for_backward(x, f, r)
        return val

    @staticmethod
    def backward(ctx, g):
        x, f, r = ctx.saved_tensors
        plan = ctx.plan
        gx = gf = None
        g = g.contiguous()
        if ctx.needs_input_grad[0] and ctx.needs_input_grad[1]:
            gx, gf = plan.adjoint_xf(r, x, f, exact=ctx.exact, scale=g)
        elif ctx.needs_input_grad[0]:
            gx = plan.adjoint_x(r * g, f, exact=ctx.exact)
        elif ctx.needs_input_grad[1]:
            gf = plan.adjoint_f(r * g, x, exact=ctx.exact)
        if gx is not None and ctx.lam:
            xc = x.contiguous()
            H, W = int(xc.shape[-2]), int(xc.shape[-1])
            _lib.call('vmbd_tv_grad', _lib.ptr(gx), _lib.ptr(xc), xc.numel() // (H * W), H, W, ctx.eps, _lib.ptr(g),
                      ctx.lam, 1, _lib.stream_ptr())
        return gx, gf, None, None, None, None, None


class OlaLoss(torch.nn.Module):
    """L(x, f) = 1/2 |B(x, f) - y|^2 + lam TV(x)."""

    def __init__(self, plan, lam=1e-3, eps=1e-3, exact=True):
        super().__init__()
        self.plan = plan
        self.lam = float(lam)
        self.eps = float(eps)
        self.exact = bool(exact)

    def _fused(self, x, f, y):
        """The operands the one-function form takes: float32 tensors on the
        plan's device, y constant (no gradient, no forward-mode tangent) and
        shaped like the result."""
        p = self.plan
        if not all(isinstance(t, torch.Tensor) and t.dtype == torch.float32 and t.device == p.device
                   for t in (x, f, y)):
            return False
        if y.requires_grad or fwAD.unpack_dual(y).tangent is not None:
            return False
        return x.dim() in (2, 3) and tuple(y.shape) == tuple(x.shape[:-2]) + p.sy

    def forward(self, x, f, y):
        if self._fused(x, f, y):
            return _LossFunction.apply(x, f, y, self.plan, self.lam, self.eps, self.exact)
        r = ola(x, f, self.plan, self.exact) - y
        out = 0.5 * (r * r).sum()
        if self.lam:
            out = out + self.lam * tv(x, self.eps)
        return out
