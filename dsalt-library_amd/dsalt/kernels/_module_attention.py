"""Autograd glue of the attention module's core: RoPE, landmark selection and weights, and
SOFT (packed) or dense attention as one differentiable function of x, q, k, v, w~ and alpha
(dsalt/modules/dsalt_attention.py:371-438, :440-487, :570-585 of the reference).

Forward: the norms pass (which rotates q and k and, for fp32 modules, writes the fp16
operands), the selection, the landmark weights and the attention. Backward: the attention's
kernels, which return dq and dk un-rotated, then the weights' backward, which adds the
norms' share to dv. Nothing of it runs as torch elementwise ops, and no rotated or cast
copy is made besides the operands the attention reads.
"""
from __future__ import annotations

import math

import torch

from .. import _hip


class _ModuleAttention(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, q, k, v, w_cont, alpha, cos, sin, cu_seqlens, k_lmk, max_seqlen, tau_lmk, tau_win, win_edge,
                dense):
        a32 = alpha.detach().to(torch.float32).contiguous()
        T, H, D = q.shape
        w32 = w_cont.detach().to(torch.float32)
        # the dense variant excludes no key from the selection (its exclusion is per query)
        w_sel = w32.new_zeros(1).expand(T) if dense else w32
        sel = _hip.SelectHybridLauncher(x.detach(), v.detach(), a32, H, w_sel, cu_seqlens, k_lmk,
                                        max_seqlen=max_seqlen, quantize=not dense,
                                        rope_k=(k.detach(), cos, sin, cu_seqlens), rope_q=q.detach())
        sel()
        weight = _hip.lmk_weights(sel.norms, a32, sel.out, sel.cu, T, v.shape[1], tau_lmk, dense)
        scale = 1.0 / math.sqrt(D)
        if dense:
            out, lse = _hip.dense_fwd(sel.q_out, sel.k_out, sel.v_out, w32, weight, scale, tau_win, win_edge)
        else:
            pos, logw = (sel.out, weight) if k_lmk > 0 else (None, None)
            out, lse = _hip.fwd(_hip.MODE_SOFT, sel.q_out, sel.k_out, sel.v_out, w32, pos, logw, sel.cu, scale, tau_win,
                                win_edge)
        # without a cast the attention's v is the input itself
        cast = sel.v_out.dtype != v.dtype
        ctx.save_for_backward(x, v, sel.q_out, sel.k_out, sel.v_out if cast else None, out, lse, w32, weight, a32,
                              sel.norms, sel.out, sel.cu, cos, sin)
        ctx.dsalt = (k_lmk, tau_lmk, tau_win, win_edge, dense, scale, q.dtype, w_cont.dtype, alpha.dtype)
        if dense:
            ctx.mark_non_differentiable(sel.out)
        else:
            ctx.mark_non_differentiable(sel.out, sel.w_out)
        return out, sel.out, sel.w_out

    @staticmethod
    def backward(ctx, grad_out, _d_pos, _d_w):
        x, v, q_r, k_r, v_c, out, lse, w32, weight, a32, norms, pos, cu, cos, sin = ctx.saved_tensors
        k_lmk, tau_lmk, tau_win, win_edge, dense, scale, od, w_dtype, a_dtype = ctx.dsalt
        v_c = v.detach() if v_c is None else v_c
        H, D, n_kv = q_r.shape[1], q_r.shape[2], k_r.shape[1]
        # grouped K/V heads: per-query-head gradients in fp32, summed over each group
        gdt = torch.float32 if (od == torch.float32 or n_kv != H) else q_r.dtype
        need_x, _, _, need_v, need_w, need_a = ctx.needs_input_grad[:6]
        if dense:
            fused = D == 64  # the dense kernels un-rotate their gradients at D = 64
            dq, dk, dv, d_weight, dw = _hip.dense_bwd(q_r, k_r, v_c, out, lse, grad_out, w32, weight, scale, tau_win,
                                                      win_edge, need_dw=need_w, grad_dtype=gdt,
                                                      rope=(cos, sin, od) if fused else None)
        else:
            fused = True
            lp, lw = (pos, weight) if k_lmk > 0 else (None, None)
            dq, dk, dv, d_weight, dw = _hip.bwd(_hip.MODE_SOFT, q_r, k_r, v_c, out, lse, grad_out, w32, lp, lw, cu, scale,
                                                tau_win, win_edge, need_dw=need_w, grad_dtype=gdt, rope=(cos, sin, od))
        dk, dv = _hip.group_sum(dk, n_kv), _hip.group_sum(dv, n_kv)
        dq, dk, dv = dq.to(od), dk.to(od), dv.to(od)
        if not fused:
            dq, dk = _hip.rope(dq, dk, cos, sin, cu, transpose=True, q_out=dq, k_out=dk)
        dx = da = None
        if d_weight is not None and (need_x or need_v or need_a):
            dx, dv_all, da = _hip.lmk_weights_bwd(d_weight, norms, a32, pos, cu, x, v, dv, tau_lmk, dense, need_x, need_v)
            dv = dv if dv_all is None else dv_all
            da = da.to(a_dtype) if need_a else None
        return (dx, dq, dk, dv, None if dw is None else dw.to(w_dtype), da, None, None, None, None, None, None, None, None,
                None)


def module_attention(x, q, k, v, w_cont, alpha, cos, sin, cu_seqlens, k_lmk: int, max_seqlen, tau_lmk: float,
                     tau_win: float, win_edge: float, dense: bool = False):
    """``(out [T, H, D] in the compute dtype, lmk_pos [H, S, k], w)`` from un-rotated q [T, H, D],
    k and v [T, n_kv, D] (operands that ``_hip.scores_supported`` and
    ``_hip.rope_operands_supported`` take), the states x [T, d], the windows w~ [T] and the
    heads' alpha; ``w`` are the quantised windows (None with ``dense``: one sequence)."""
    return _ModuleAttention.apply(x, q, k, v, w_cont, alpha, cos, sin, cu_seqlens, k_lmk, max_seqlen, tau_lmk, tau_win,
                                  win_edge, dense)
