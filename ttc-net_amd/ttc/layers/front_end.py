"""The layer's front-end between ``in_proj`` and the solver (``ttc/layers/ttc_layer.py:110-135``):
the split of the projection, ``l2norm`` / softplus / clamp and the log-discounts.

:func:`front_end` takes the projection ``[N, row]`` and returns ``(A_diag, coeff_B, coeff_Q, R_inv,
coeff_Qf, log_gamma_A, log_gamma_B, log_gamma_Q, h0)``.  fp32 CUDA projections go through one kernel
each way (``ttc_lqr_front_end`` / ``_backward``, contiguous outputs); anything else, and any call under a
functorch transform, forward-mode AD, a dispatch mode or tracing, runs :func:`front_end_torch`, the same
formulas as torch operators.  The backward differentiates :func:`front_end_torch` when it is itself
recorded (``create_graph=True``) or so observed (batched gradients), so second derivatives of the
front-end are what autograd gives for the operators.
"""
from __future__ import annotations

import torch
import torch.nn.functional as F

from ..solvers._lib import lib, check

__all__ = ["front_end", "front_end_torch", "l2norm"]


def l2norm(x: torch.Tensor, eps: float = 1e-6) -> torch.Tensor:
    xf = x.float()
    return (xf * torch.rsqrt((xf * xf).sum(-1, keepdim=True) + eps)).to(x.dtype)


def front_end_torch(proj: torch.Tensor, bias: torch.Tensor | None, dims):
    H, hd, ud, rb, rq = dims
    head = [hd, hd, ud, rq, 1 + ud + hd]
    heads, coeff_B, coeff_Q = torch.split(proj, [sum(head) * H, rb, rq], dim=-1)
    h0, A_diag, R_inv_diag, coeff_Qf, log_gammas = torch.split(heads.reshape(-1, H, sum(head)), head, dim=-1)
    A_diag = l2norm(A_diag)
    coeff_B, coeff_Q, coeff_Qf = l2norm(coeff_B), l2norm(F.softplus(coeff_Q)), l2norm(F.softplus(coeff_Qf))
    R_inv_diag = torch.clamp(l2norm(F.softplus(R_inv_diag)), min=1e-6)
    if bias is not None:
        log_gammas = -F.softplus(log_gammas) - F.relu(-bias[None, None, :])
    else:
        log_gammas = -F.softplus(log_gammas)
    lgA, lgB, lgQ = torch.split(log_gammas, [1, ud, hd], dim=-1)
    return A_diag, coeff_B, coeff_Q, R_inv_diag, coeff_Qf, lgA.squeeze(-1), lgB, lgQ, h0


class _FrontEndFunc(torch.autograd.Function):

    @staticmethod
    def forward(ctx, proj, bias, dims):
        H, hd, ud, rb, rq = dims
        N = proj.shape[0]
        ctx.dims = dims
        ctx.set_materialize_grads(False)
        ctx.save_for_backward(proj, bias)
        p = proj.detach().contiguous()
        b = None if bias is None else bias.detach().contiguous()
        E = lambda *s: torch.empty(*s, device=p.device, dtype=torch.float32)  # noqa: E731
        out = (E(N, H, hd), E(N, rb), E(N, rq), E(N, H, ud), E(N, H, rq), E(N, H), E(N, H, ud), E(N, H, hd),
               E(N, H, hd))
        with torch.cuda.device(p.device):
            rc = lib.ttc_lqr_front_end(p.data_ptr(), None if b is None else b.data_ptr(), N, H, hd, ud, rb, rq,
                                       *[t.data_ptr() for t in out],
                                       torch.cuda.current_stream(p.device).cuda_stream)
        check(rc, "ttc_lqr_front_end")
        return out

    @staticmethod
    def backward(ctx, *grads):
        proj, bias = ctx.saved_tensors
        need_proj, need_bias = ctx.needs_input_grad[:2]
        if all(g is None for g in grads):
            return None, None, None
        recorded = torch.is_grad_enabled()
        if recorded or _traced(proj, bias, *grads):  # differentiable operators, seen one by one
            with torch.enable_grad():
                if not recorded:
                    proj, bias = (t if t is None else t.detach().requires_grad_() for t in (proj, bias))
                out = front_end_torch(proj, bias, ctx.dims)
                pairs = [(o, g) for o, g in zip(out, grads) if g is not None]
                wrt = [t for t, need in ((proj, need_proj), (bias, need_bias)) if need]
                got = iter(torch.autograd.grad([o for o, _ in pairs], wrt, [g for _, g in pairs],
                                               create_graph=recorded, allow_unused=True))
            return next(got) if need_proj else None, next(got) if need_bias else None, None
        H, hd, ud, rb, rq = ctx.dims
        N = proj.shape[0]
        d_proj = d_bias = None
        if need_proj:
            p = proj.contiguous()
            gs = [None if g is None else g.to(torch.float32).contiguous() for g in grads]
            d_proj = torch.empty_like(p)
            with torch.cuda.device(p.device):
                rc = lib.ttc_lqr_front_end_backward(p.data_ptr(), N, H, hd, ud, rb, rq,
                                                    *[None if g is None else g.data_ptr() for g in gs],
                                                    d_proj.data_ptr(),
                                                    torch.cuda.current_stream(p.device).cuda_stream)
            check(rc, "ttc_lqr_front_end_backward")
        if need_bias:
            zero = lambda g, n: bias.new_zeros(n) if g is None else g.reshape(N * H, n).sum(0)  # noqa: E731
            d_bias = torch.cat([zero(grads[5], 1), zero(grads[6], ud), zero(grads[7], hd)])
            d_bias = d_bias.masked_fill(bias >= 0, 0.0)  # relu's gradient: 0 where it is off, NaN passes
        return d_proj, d_bias, None


def _traced(*xs) -> bool:
    """Whether operators are observed one by one (functorch transforms, batched gradients, forward-mode
    tangents, tracing and compilation, dispatch modes such as ``make_fx``'s, tensor subclasses such as fake
    tensors): none of these sees the kernel."""
    if torch.compiler.is_compiling():  # first: a full-graph compilation can trace none of the rest
        return True
    return (any(type(x) not in (torch.Tensor, torch.nn.Parameter) or not torch._C._has_storage(x)
                for x in xs if x is not None)
            or torch._C._are_functorch_transforms_active() or torch._C._len_torch_dispatch_stack() > 0
            or torch.autograd.forward_ad._current_level >= 0 or torch.jit.is_tracing())


def front_end(proj: torch.Tensor, bias: torch.Tensor | None, dims):
    """``dims = (heads, h_dim, u_dim, b_rank, q_rank)``.  The kernel takes exactly the sizes that these give; the
    operators broadcast any other bias, or raise."""
    H, hd, ud, rb, rq = dims
    if not _traced(proj, bias) and proj.is_cuda and proj.dtype == torch.float32 and (
            proj.dim() == 2 and proj.shape[1] == (3 * hd + 2 * ud + rq + 1) * H + rb + rq) and (
            bias is None or (bias.device == proj.device and bias.dtype == torch.float32
                             and bias.shape == (1 + ud + hd,))):
        return _FrontEndFunc.apply(proj, bias, dims)
    return front_end_torch(proj, bias, dims)
