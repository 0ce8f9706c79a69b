"""DSALT inference attention (HARD selectors) on the gfx950 HIP kernels.

Drop-in for dsalt/kernels/dsalt_triton_attn.py: same entry point
``dsalt_triton_attention(q, k, v, lmk_indices, lmk_bias, w_sizes, cu_seqlens)`` and the
same ``DSALTAttentionFunction`` (returns fp32 output, gradients in q's dtype; fp32
inputs compute as fp16, dsalt_triton_attn.py:259-328). The module name is kept for
import compatibility; nothing here uses Triton.

Semantics (dsalt_triton_attn.py:69-169): query i of a sequence attends to keys
``[i - w + 1, i]`` with ``w = max(1, trunc(w_sizes[i]))`` and to landmark slot p when
``0 <= p <= i - w``, with logit ``q.k / sqrt(D) + lmk_bias[h, s, slot]``.
"""
from __future__ import annotations

import functools

import torch

from .. import _hip
from . import _sparse
from .autotune import autotune_blocks, get_tuned_config  # noqa: F401  (re-exports)
from .dsalt_triton_bwd import dsalt_triton_backward  # noqa: F401
from .landmark_tokens_ker import hybrid_scores_per_head  # noqa: F401
from .selectors import (  # noqa: F401  (re-exported like the reference, :18-24)
    _build_landmark_kv,
    _build_seq_block_map,
    _compute_landmark_indices,
    _score_block,
    _seq_meta,
)


class DSALTAttentionFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v, lmk_indices, lmk_bias, w_sizes, cu_seqlens):
        return _sparse._forward(ctx, _hip.MODE_HARD, q, k, v, lmk_indices, lmk_bias, w_sizes,
                                cu_seqlens, 1.0, 4.0, out_f32=True)

    @staticmethod
    def backward(ctx, grad_out):
        dq, dk, dv, d_bias, _ = _sparse._backward(ctx, grad_out, need_dw=False)
        return dq, dk, dv, None, d_bias, None, None


def _dynamo_opaque(fn):
    """fn as a call that torch.compile does not trace into; outside of it, fn itself (the
    disabled wrapper's frame switch costs microseconds on every call)."""
    disable = getattr(getattr(torch, "_dynamo", None), "disable", None)
    if disable is None:
        return fn
    opaque = disable(fn)

    @functools.wraps(fn)
    def call(*args, **kwargs):
        return opaque(*args, **kwargs) if torch.compiler.is_compiling() else fn(*args, **kwargs)

    return call


@_dynamo_opaque
def dsalt_triton_attention(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    lmk_indices: torch.Tensor,
    lmk_bias: torch.Tensor,
    w_sizes: torch.Tensor,
    cu_seqlens: torch.Tensor,
) -> torch.Tensor:
    """HARD DSALT attention over packed ``[T, H, D]`` q/k/v; returns fp32 ``[T, H, D]``."""
    if _sparse.no_graph(q, k, v, lmk_indices, lmk_bias, w_sizes, cu_seqlens):
        return _sparse._forward(None, _hip.MODE_HARD, q, k, v, lmk_indices, lmk_bias, w_sizes, cu_seqlens, 1.0, 4.0,
                                out_f32=True)
    return DSALTAttentionFunction.apply(q, k, v, lmk_indices, lmk_bias, w_sizes, cu_seqlens)
