"""Autograd glue of the transformer block's own passes: residual add with the RMSNorm after it,
residual add alone, and the SwiGLU feed-forward as one function each
(dsalt/modules/dsalt_transformer.py:10-21, :81-84 of the reference).
"""
from __future__ import annotations

import functools

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.autograd import forward_ad

from .. import _hip


def plain(*mods: nn.Module) -> bool:
    """Whether calling these modules does nothing but their class's forward: no hooks on them
    or on all modules, no forward set on the instance."""
    g = nn.modules.module
    if (g._global_forward_hooks or g._global_forward_pre_hooks or g._global_backward_hooks
            or g._global_backward_pre_hooks):
        return False
    return not any(m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks
                   or "forward" in m.__dict__ for m in mods)


def eager(*ts: torch.Tensor) -> bool:
    """Whether these tensors are being computed with directly: not traced or compiled, under no
    functorch transform or forward-mode level, and of no tensor subclass. Otherwise torch's
    own ops run, which those understand."""
    if torch.compiler.is_compiling() or torch.jit.is_tracing() or torch._C._are_functorch_transforms_active():
        return False
    return forward_ad._current_level < 0 and all(type(t) in (torch.Tensor, nn.Parameter) for t in ts)


def autocast_dtype(x: torch.Tensor) -> torch.dtype:
    """Element type of a projection's result for x: autocast's where it is on."""
    return torch.get_autocast_dtype("cuda") if torch.is_autocast_enabled("cuda") else x.dtype


def autocast_state() -> tuple[bool, torch.dtype]:
    """Autocast as it is here, for ``autocast_as`` in a backward."""
    return torch.is_autocast_enabled("cuda"), torch.get_autocast_dtype("cuda")


def autocast_as(state: tuple[bool, torch.dtype]):
    return torch.autocast("cuda", dtype=state[1], enabled=state[0])


def without_autocast(backward):
    """A backward whose operands have their types already: an autocast that is on where it runs
    (a backward called inside one, maybe of another type than the forward's) changes nothing."""
    @functools.wraps(backward)
    def call(ctx, *grads):
        if not torch.is_autocast_enabled("cuda"):
            return backward(ctx, *grads)
        with torch.autocast("cuda", enabled=False):
            return backward(ctx, *grads)

    return call


def graph_grads(fn, inputs, dys):
    """Differentiable gradients of fn(*inputs), with the upstream gradients dys of its outputs (None:
    none), with respect to the inputs that require one (else None). fn sees aliases of the
    inputs, so that one which depends on another (v on x) gives its own share only."""
    with torch.enable_grad():
        alias = [t.view_as(t) if t is not None and t.requires_grad else t for t in inputs]
        live = [t for t in alias if t is not None and t.requires_grad]
        pairs = [(y, dy.to(y.dtype)) for y, dy in zip(fn(*alias), dys) if dy is not None and y.requires_grad]
        got = iter(torch.autograd.grad([y for y, _ in pairs], live, [d for _, d in pairs], create_graph=True,
                                       allow_unused=True))
        return [next(got) if t is not None and t.requires_grad else None for t in inputs]


def valued(t: torch.Tensor, value: torch.Tensor) -> torch.Tensor:
    """t's graph at the value that the forward had (a parameter may have changed since)."""
    return value.to(t.dtype) + (t - t.detach())


class _AddNorm(torch.autograd.Function):
    """(x_out, y): the sum (x itself without h) and its norm, in x's dtype or only rounded to
    `cast` (cast_only); with both, y_cast is a third output that takes no gradient."""

    @staticmethod
    def forward(ctx, x, h, weight, eps, cast, cast_only):
        ctx.set_materialize_grads(False)
        xd = x.detach()
        s, y, y_cast, rstd = _hip.norm_train(xd, None if h is None else h.detach(), weight.detach(), eps,
                                             not cast_only, cast)
        ctx.save_for_backward(x if s is None else s, weight, rstd)
        ctx.dsalt = (None if h is None else h.dtype), x.dtype, eps
        s = x.view_as(x) if s is None else s
        if cast_only:
            return s, y_cast
        if cast is None:
            return s, y
        ctx.mark_non_differentiable(y_cast)
        return s, y, y_cast

    @staticmethod
    def backward(ctx, ds, dy, *_):
        x, weight, rstd = ctx.saved_tensors
        h_dtype, x_dtype, eps = ctx.dsalt
        need_x, need_h, need_w = ctx.needs_input_grad[:3]
        if dy is None:
            dh = ds.to(h_dtype) if need_h and ds is not None else None
            return ds if need_x else None, dh, None, None, None, None
        if torch.is_grad_enabled():  # a graph of the backward is wanted: torch's own ops
            dx, dw = graph_grads(lambda x, w: (F.rms_norm(x, x.shape[-1:], w, eps),), (x, weight), (dy,))
            ds = dx if ds is None else ds if dx is None else ds + dx
            dh = ds.to(h_dtype) if need_h else None
            return ds if need_x else None, dh, dw if need_w else None, None, None, None
        dy = _hip.aligned_rows(dy)
        ds = None if ds is None else _hip.aligned_rows(ds)
        same = need_h and h_dtype == x_dtype  # the branch's gradient is then the residual's
        dx, dh, dw = _hip.norm_train_bwd(x.detach(), weight.detach(), rstd, dy, ds,
                                         h_dtype if need_h and not same else None, need_x or same, need_w)
        return dx if need_x else None, dx if same else dh, dw, None, None, None


class _Add(torch.autograd.Function):
    """fp32 x + 16-bit h in one pass."""

    @staticmethod
    def forward(ctx, x, h):
        ctx.h_dtype = h.dtype
        return _hip.norm_train(x.detach(), h.detach(), None, 0.0)[0]

    @staticmethod
    def backward(ctx, dy):
        return dy if ctx.needs_input_grad[0] else None, dy.to(ctx.h_dtype) if ctx.needs_input_grad[1] else None


class _SwiGLU(torch.autograd.Function):
    """down(silu(gate(x)) * up(x)): one GEMM for gate and up, two for their gradients."""

    @staticmethod
    def forward(ctx, x, wg, wu, wd, dtype):
        f, d = wg.shape
        xb = x.detach().reshape(-1, d)
        xb = xb if xb.dtype == dtype else xb.to(dtype)
        if wg.dtype == dtype:
            w_gu, w_d = torch.cat([wg.detach(), wu.detach()]), wd.detach()
        else:
            w_gu = torch.empty((2 * f, d), device=x.device, dtype=dtype)
            w_gu[:f].copy_(wg.detach())
            w_gu[f:].copy_(wu.detach())
            w_d = wd.detach().to(dtype)
        gu = torch.mm(xb, w_gu.t())
        a = _hip.swiglu_rows(gu)
        # not a view of the GEMM's result: torch lets no one modify a view from a function in place
        y = torch.empty((*x.shape[:-1], w_d.shape[0]), device=x.device, dtype=dtype)
        torch.mm(a, w_d.t(), out=y.view(-1, w_d.shape[0]))
        cast = xb.dtype != x.dtype
        # the weights are saved where a gradient needs them, as three linears would: changed in place
        # before the backward they are refused then (the backward itself takes w_gu and w_d)
        need_x, need_g, need_u = ctx.needs_input_grad[:3]
        saved = (wg, wu) if need_x else (None, None)
        ctx.save_for_backward(x, *saved, wd if need_x or need_g or need_u else None, gu, a, w_gu, xb if cast else None,
                              w_d if w_d.dtype != wd.dtype else None)
        ctx.dsalt_params = wg, wu, wd  # for a graph of the backward: the parameters, unchecked
        return y

    @staticmethod
    @without_autocast
    def backward(ctx, dy):
        x, _, _, wd, gu, a, w_gu, xb, w_d = ctx.saved_tensors
        if torch.is_grad_enabled():  # a graph of the backward is wanted: torch's own ops
            def ffn(*inputs):
                xc, g, u, d = (t.to(gu.dtype) for t in inputs)
                xc, f = xc.reshape(-1, xc.shape[-1]), g.shape[0]
                h = F.silu(valued(F.linear(xc, g), gu[:, :f])) * valued(F.linear(xc, u), gu[:, f:])
                return F.linear(h, d).view(dy.shape),

            return *graph_grads(ffn, (x, *ctx.dsalt_params), (dy,)), None
        shape, x_dtype, w_dtype, f = x.shape, x.dtype, ctx.dsalt_params[0].dtype, a.shape[1]
        xb = (x.detach() if xb is None else xb).reshape(-1, shape[-1])
        dy = dy.reshape(-1, dy.shape[-1])
        need_x, need_g, need_u, need_d = ctx.needs_input_grad[:4]
        dx = dg = du = dwd = None
        if need_d:
            dwd = torch.mm(dy.t(), a).to(w_dtype)
        if need_x or need_g or need_u:
            dgu = _hip.swiglu_rows(gu, torch.mm(dy, wd.detach() if w_d is None else w_d))
            if need_g and need_u:
                dg, du = torch.mm(dgu.t(), xb).to(w_dtype).split(f)
            else:
                dg = torch.mm(dgu[:, :f].t(), xb).to(w_dtype) if need_g else None
                du = torch.mm(dgu[:, f:].t(), xb).to(w_dtype) if need_u else None
            if need_x:
                dx = torch.mm(dgu, w_gu).view(shape).to(x_dtype)
        return dx, dg, du, dwd, None


def add_norm(x, h, norm, cast=None, cast_only=False):
    """``(x + h, norm(x + h)[, norm rounded to cast])``; h None: ``(x, norm(x)[, ...])``. Operands as
    _hip.norm_train_supported and norm_train_branch_supported check them."""
    return _AddNorm.apply(x, h, norm.weight, norm.eps, cast, cast_only)


def residual_add(x, h):
    """``x + h``; an fp32 stream and a 16-bit branch in one HIP pass, else torch's add."""
    if x.dtype == torch.float32 and h.dtype != x.dtype and eager(x, h) and x.is_cuda and x.shape[-1] % 8 == 0 and \
            8 <= x.shape[-1] <= _hip.RMS_NORM_MAX_DIM and x.numel() and _hip._rows_aligned(x) and \
            _hip.norm_train_branch_supported(x, h):
        return _Add.apply(x, h)
    return x + h


def swiglu_supported(ffn, x: torch.Tensor) -> bool:
    """Whether the SwiGLUFFN `ffn` runs on x as one function: plain nn.Linear projections
    without bias, of one dtype that is x's own, or fp32 under a 16-bit autocast (x fp32 or
    already rounded)."""
    lin = (ffn.gate_proj, ffn.up_proj, ffn.down_proj)
    if not (eager(x, *(m.weight for m in lin)) and x.is_cuda and x.dim() >= 2 and x.numel() and all(type(m) is nn.Linear for m in lin) and plain(*lin)):
        return False
    wg, wu, wd = (m.weight for m in lin)
    if any(m.bias is not None for m in lin) or any(w.dtype != wg.dtype or w.device != x.device for w in (wg, wu, wd)):
        return False
    f, d = wg.shape
    if wu.shape != (f, d) or wd.shape[1] != f or x.shape[-1] != d or f % 8 or not x.is_contiguous():
        return False
    dt = autocast_dtype(x)
    if dt not in (torch.bfloat16, torch.float16, torch.float32):
        return False
    return wg.dtype == dt == x.dtype or (wg.dtype == torch.float32 and dt != torch.float32 and x.dtype in (dt, torch.float32))


def swiglu_ffn(ffn, x: torch.Tensor) -> torch.Tensor:
    return _SwiGLU.apply(x, ffn.gate_proj.weight, ffn.up_proj.weight, ffn.down_proj.weight, autocast_dtype(x))
