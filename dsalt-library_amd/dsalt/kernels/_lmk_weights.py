"""Autograd glue of the landmark selection and its differentiable weights.

The selection is detached; the weight log(max(sigmoid(s / tau_lmk), 1e-20)) of each selected
landmark carries gradients to x, to the value projection v and to the per-head balance
alpha through the hybrid score s (dsalt/modules/dsalt_attention.py:403-438, :457-487 of the
reference). The HIP norms pass and the selection give the landmarks; ``dsalt_lmk_weights``
gives their weights from the same norms and statistics, and its backward is two launches.
``v`` is also returned, so that the attention's gradient of v arrives here and the norms'
share is added to it in the pass that forms it.
"""
from __future__ import annotations

import torch

from .. import _hip
from ._block_train import autocast_as, autocast_state, graph_grads
from .landmark_tokens_ker import hybrid_scores_from_v


def torch_weights(x, v, alpha, pos, cu, tau: float, table: bool) -> torch.Tensor:
    """The weights of ``landmark_weights`` at the landmarks ``pos`` in torch's ops, for a graph of
    the backward."""
    T, (H, S, k) = x.shape[0], pos.shape
    scores = hybrid_scores_from_v(x, v, alpha, H)[0]
    if table:
        sel = torch.zeros(H, T + 1, dtype=torch.bool, device=x.device)
        sel.scatter_(1, torch.where(pos[:, 0] >= 0, pos[:, 0], T), True)
        return torch.log(torch.sigmoid(scores.float() / tau).clamp(min=1e-20)).t().where(sel[:, :T], float("-inf"))
    tok = cu[:-1].long().clamp(0, T - 1).view(1, S, 1) + pos.clamp(min=0)
    s = scores.t().gather(1, tok.view(H, S * k)).view(H, S, k)
    return torch.sigmoid(s / tau).clamp(min=1e-20).log().masked_fill(pos < 0, float("-inf"))


class _LandmarkWeights(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, v, alpha, w_cont, cu_seqlens, k_lmk, max_seqlen, tau, table):
        ctx.set_materialize_grads(False)
        a32 = alpha.detach().to(torch.float32).contiguous()
        sel = _hip.SelectHybridLauncher(x.detach(), v.detach(), a32, a32.shape[0], w_cont.detach(), cu_seqlens, k_lmk,
                                        max_seqlen=max_seqlen, quantize=not table)
        sel()
        weight = _hip.lmk_weights(sel.norms, a32, sel.out, sel.cu, x.shape[0], v.shape[1], tau, table)
        ctx.save_for_backward(x, v, alpha, sel.norms, sel.out, sel.cu)
        ctx.dsalt_tau, ctx.dsalt_table, ctx.dsalt_autocast = tau, table, autocast_state()
        ctx.mark_non_differentiable(sel.out, *(() if table else (sel.w_out,)))
        return v.view_as(v), weight, sel.out, sel.w_out

    @staticmethod
    def backward(ctx, dv_in, d_weight, _d_pos, _d_w):
        if d_weight is None:
            return None, dv_in, None, None, None, None, None, None, None
        x, v, alpha, norms, pos, cu = ctx.saved_tensors
        need_x, need_v, need_a = ctx.needs_input_grad[:3]
        if torch.is_grad_enabled():  # a graph of the backward is wanted: torch's own ops
            with autocast_as(ctx.dsalt_autocast):
                dx, dv, da = graph_grads(lambda *t: (torch_weights(*t, pos, cu, ctx.dsalt_tau, ctx.dsalt_table),),
                                         (x, v, alpha), (d_weight,))
            dv = dv_in if dv is None else dv if dv_in is None else dv_in + dv
            return dx, dv, da, None, None, None, None, None, None
        a32 = alpha.detach().to(torch.float32).contiguous()
        dx, dv, da = _hip.lmk_weights_bwd(d_weight, norms, a32, pos, cu, x, v, dv_in, ctx.dsalt_tau, ctx.dsalt_table,
                                          need_x, need_v)
        return dx, dv, da.to(alpha.dtype) if need_a else None, None, None, None, None, None, None


def landmark_weights(x, v, alpha, w_cont, cu_seqlens, k_lmk: int, max_seqlen, tau: float, table: bool = False):
    """``(v, weights, lmk_pos [H, S, k], w)``: the landmarks of packed x [T, d] selected by the
    hybrid score from v [T, n_kv, D] (``_hip.scores_supported`` operands), outside the
    windows floor(``w_cont``) (returned quantised as ``w``), with their weights [H, S, k]
    (-inf in empty slots). ``table``: one sequence, ``w_cont`` taken as it is (``w`` is
    None), the weights as the [H, T] table (-inf off the landmarks)."""
    return _LandmarkWeights.apply(x, v, alpha, w_cont, cu_seqlens, k_lmk, max_seqlen, tau, table)
