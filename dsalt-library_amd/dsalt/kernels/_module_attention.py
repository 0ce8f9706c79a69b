"""Autograd glue of the attention module's core: q/k/v projections, window gate, RoPE,
landmark selection and weights, and SOFT (packed) or dense attention as one differentiable
function of the states and the parameters (dsalt/modules/dsalt_attention.py:270-284,
:371-438, :440-487, :566-585 of the reference).

Forward: one GEMM against the three projection weights concatenated; the norms pass, which
also forms the gate's logits and windows, rotates q and k in place and, for fp32 modules,
writes the fp16 operands; the selection; the landmark weights; the attention. Backward: the
attention's kernels write dq, dk (un-rotated) and dv into one [T, d + 2 kv] buffer, the
norms' share is added to dv, two GEMMs give the weights' gradients and dx, and one pass adds
the norm and gate shares to dx and sums the gate's gradients.
"""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from .. import _hip
from ._block_train import autocast_as, autocast_state, graph_grads, valued, without_autocast
from ._lmk_weights import torch_weights


class _ModuleAttention(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, wq, wk, wv, wg, bg, alpha_w, cos, sin, cu_seqlens, opt, x_cast):
        ctx.set_materialize_grads(False)  # no zero gradients of the outputs that take none
        cdt, H, n_kv, D = opt["dtype"], opt["n_heads"], opt["n_kv_heads"], opt["head_dim"]
        T, dense, k_lmk = x.shape[0], opt["dense"], opt["k_lmk"]
        xd = x.detach()
        xb = xd if xd.dtype == cdt else xd.to(cdt) if x_cast is None else x_cast.detach()
        ws = [w.detach() for w in (wq, wk, wv)]
        if wq.dtype == cdt:
            w_cat = torch.cat(ws)
        else:
            w_cat = torch.empty((sum(w.shape[0] for w in ws), x.shape[1]), device=x.device, dtype=cdt)
            for dst, w in zip(w_cat.split([w.shape[0] for w in ws]), ws):
                dst.copy_(w)
        qkv = torch.mm(xb, w_cat.t())
        q, k, v = _split(qkv, H, n_kv, D)
        a32 = torch.sigmoid(alpha_w.detach()).to(torch.float32)
        sel = _hip.SelectHybridLauncher(
            xd, v, a32, H, None, cu_seqlens, k_lmk, max_seqlen=opt["max_seqlen"], quantize=not dense,
            rope_k=(k, cos, sin, cu_seqlens), rope_q=q, window=(wg.detach(), None if bg is None else bg.detach(), cdt,
                                                                opt["n_min"], opt["n_max"]), free_windows=dense)
        sel()
        weight = _hip.lmk_weights(sel.norms, a32, sel.out, sel.cu, T, n_kv, opt["tau_lmk"], dense)
        scale = 1.0 / math.sqrt(D)
        if dense:
            out, lse = _hip.dense_fwd(sel.q_out, sel.k_out, sel.v_out, sel.win_out, weight, scale, opt["tau_win"],
                                      opt["win_edge"])
        else:
            pos, logw = (sel.out, weight) if k_lmk > 0 else (None, None)
            out, lse = _hip.fwd(_hip.MODE_SOFT, sel.q_out, sel.k_out, sel.v_out, sel.win_out, pos, logw, sel.cu, scale,
                                opt["tau_win"], opt["win_edge"])
        cast = cdt == torch.float32  # separate fp16 operands; otherwise q and k were rotated in place
        ops = (sel.q_out, sel.k_out, sel.v_out) if cast else (None, None, None)
        # the weights are saved where x takes a gradient, as four linears would: changed in place
        # before the backward they are refused then (the backward itself takes w_cat and,
        # for dx, wg)
        saved = (wq, wk, wv, wg) if ctx.needs_input_grad[0] else (None,) * 4
        ctx.save_for_backward(x, None if xb is xd else xb, qkv, *ops, w_cat, out, lse, sel.win_logit, sel.win_out,
                              weight, a32, sel.norms, sel.out, sel.cu, cos, sin, *saved)
        ctx.dsalt = opt, scale, wq.dtype, alpha_w.dtype
        ctx.dsalt_gate = None if ctx.needs_input_grad[0] else wg.detach()
        # for a graph of the backward only: the parameters themselves, unchecked
        ctx.dsalt_params, ctx.dsalt_autocast = (wq, wk, wv, wg, bg, alpha_w), autocast_state()
        if dense:
            ctx.mark_non_differentiable(sel.out, sel.win_out)
        else:
            ctx.mark_non_differentiable(sel.out, sel.win_out, sel.w_out)
        return out, sel.out, sel.win_out, sel.w_out

    @staticmethod
    @without_autocast
    def backward(ctx, grad_out, *_):
        if grad_out is None:
            return (None,) * 12
        (x, xb, qkv, q_r, k_r, v_r, w_cat, out, lse, logit, w32, weight, a32, norms, pos, cu, cos, sin,
         _, _, _, wg) = ctx.saved_tensors
        wg = ctx.dsalt_gate if wg is None else wg
        opt, scale, w_dtype, a_dtype = ctx.dsalt
        H, n_kv, D, dense, od = opt["n_heads"], opt["n_kv_heads"], opt["head_dim"], opt["dense"], qkv.dtype
        T, grouped = x.shape[0], n_kv != H
        xb = x.detach() if xb is None else xb
        need_x, *need_w = ctx.needs_input_grad[:4]
        need_gate = ctx.needs_input_grad[4] or ctx.needs_input_grad[5]
        q, k, v = _split(qkv, H, n_kv, D)
        if q_r is None:
            q_r, k_r, v_r = q, k, v
        dqkv = torch.empty_like(qkv)
        dq, dk, dv = _split(dqkv, H, n_kv, D)
        # grouped K/V heads: per-query-head gradients in fp32, summed over each group below
        gdt, grads = (torch.float32, (dq, None, None)) if grouped else (od, (dq, dk, dv))
        fused = not dense or D == 64  # the dense kernels un-rotate their gradients at D = 64
        rope = (cos, sin, od) if fused else None
        if dense:
            _, dk_h, dv_h, d_weight, dw = _hip.dense_bwd(q_r, k_r, v_r, out, lse, grad_out, w32, weight, scale,
                                                            opt["tau_win"], opt["win_edge"], True, gdt, rope, grads)
        else:
            lp, lw = (pos, weight) if opt["k_lmk"] > 0 else (None, None)
            _, dk_h, dv_h, d_weight, dw = _hip.bwd(_hip.MODE_SOFT, q_r, k_r, v_r, out, lse, grad_out, w32, lp, lw, cu,
                                                      scale, opt["tau_win"], opt["win_edge"], True, gdt, rope, grads)
        if torch.is_grad_enabled():
            if grouped:
                dk, dv = _hip.group_sum_pair(dk_h, dv_h, n_kv, od)
            if not fused:
                _hip.rope(dq, dk, cos, sin, cu, transpose=True, q_out=dq, k_out=dk)
            return (*_graph_grads(ctx, x, v, pos, cu, logit, a32, (dq, dk, dv, dw, d_weight)), *[None] * 5)
        g = _hip.ModuleGrads(x.detach(), v, norms, a32, pos, cu, weight if d_weight is None else d_weight,
                             opt["tau_lmk"], dense)
        d_alpha = g.values(dk_h, dv_h, dk, dv, alpha_sigmoid=True)
        if not fused:
            _hip.rope(dq, dk, cos, sin, cu, transpose=True, q_out=dq, k_out=dk)
        dws = [None, None, None]
        if all(need_w):
            d_cat = torch.mm(dqkv.t(), xb)
            dws = (d_cat if w_dtype == od else d_cat.to(w_dtype)).split([H * D, n_kv * D, n_kv * D])
        elif any(need_w):
            parts = dqkv.split([H * D, n_kv * D, n_kv * D], 1)
            dws = [torch.mm(p.t(), xb).to(w_dtype) if n else None for p, n in zip(parts, need_w)]
        dx = dwg = dbg = None
        if need_x or need_gate:
            dx_in = torch.mm(dqkv, w_cat) if need_x else None
            dx, dwg, dbg = g.states(dx_in, need_x, (wg, logit, dw, od, opt["n_min"], opt["n_max"]))
        if not ctx.needs_input_grad[5]:
            dbg = None
        if not ctx.needs_input_grad[6] or not (dense or opt["k_lmk"] > 0):
            d_alpha = None  # without landmark slots alpha takes no part
        return (dx, *dws, dwg if ctx.needs_input_grad[4] else None, dbg,
                None if d_alpha is None else d_alpha.to(a_dtype), *[None] * 5)


def _graph_grads(ctx, x, v_saved, pos, cu, logit, a32, core):
    """The gradients of x and the parameters with a graph, from those of the attention's operands
    (``core``: un-rotated dq, dk, dv, the windows' and the landmark weights'), which are
    constants in it, as sparse_attention's are: projections, windows and weights in torch's
    ops, on the values that the forward had."""
    opt = ctx.dsalt[0]
    dq, dk, dv, dw, d_weight = core

    def operands(x, wq, wk, wv, wg, bg, alpha_w):
        v = valued(F.linear(x, wv).view(v_saved.shape), v_saved)
        gate = torch.sigmoid(valued(F.linear(x, wg, bg).squeeze(-1), logit))
        yield from (F.linear(x, wq), F.linear(x, wk), v, opt["n_min"] + gate * (opt["n_max"] - opt["n_min"]))
        if d_weight is not None:
            yield torch_weights(x, v, valued(torch.sigmoid(alpha_w), a32), pos, cu, opt["tau_lmk"], opt["dense"])

    with autocast_as(ctx.dsalt_autocast):
        got = graph_grads(operands, (x, *ctx.dsalt_params), (dq.flatten(1), dk.flatten(1), dv, dw, d_weight))
    return [g if n else None for g, n in zip(got, ctx.needs_input_grad)]


def _split(qkv: torch.Tensor, H: int, n_kv: int, D: int):
    """q [T, H, D], k and v [T, n_kv, D]: the column views of qkv [T, (H + 2 n_kv) D]."""
    T = qkv.shape[0]
    q, k, v = qkv.split([H * D, n_kv * D, n_kv * D], 1)
    return q.view(T, H, D), k.view(T, n_kv, D), v.view(T, n_kv, D)


def module_attention(x, q_proj, k_proj, v_proj, win_gate, alpha_w, cos, sin, cu_seqlens, opt: dict, x_cast=None):
    """``(out [T, H, D] in the compute dtype, lmk_pos [H, S, k], w~ [T], quantised w or None)`` of
    packed states x [T, d]. The four projections are plain nn.Linear modules (q, k and v
    without bias); ``opt``: dtype (of the projections' results), n_heads, n_kv_heads,
    head_dim, k_lmk, max_seqlen, tau_lmk, tau_win, win_edge, n_min, n_max, dense (one
    sequence, the dense variant). ``x_cast``: x rounded to dtype, if the caller has it.
    Operands: as DSALTAttention._one_function checks them."""
    return _ModuleAttention.apply(x, q_proj.weight, k_proj.weight, v_proj.weight, win_gate.weight, win_gate.bias, alpha_w,
                                  cos, sin, cu_seqlens, opt, x_cast)
