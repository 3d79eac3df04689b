"""Fused split + per-head RMSNorm of the qkv projection (autograd Function over libsa2).

Does in one kernel what HigherOrderAttention.forward does between the ``to_qkv``
projection and the attention call when there are two key/value sets and heads are not
moved in front of the sequence (simplicial_mha.py:116-127 of the reference): split into
q | k | v, unflatten heads with channel order ``(head, set, d)``, chunk the sets apart and
apply the five ``RMSNorm(dim_head)`` modules.
"""
from __future__ import annotations

import torch
from torch.autograd import Function

from . import _native


class FusedQKVNorm(Function):
    """``apply(qkv, wq, wk1, wk2, wv1, wv2, heads, kv_heads, dim_head, eps) -> q, k1, k2, v1, v2``.

    ``qkv``: (b, n, (heads + 4 kv_heads) * dim_head) bf16 on the GPU; the weights are the
    ``weight`` tensors of the five RMSNorm modules (bf16, ``(dim_head,)``) or ``None``.
    Outputs are contiguous (b, n, h, dim_head).
    """

    @classmethod
    def apply(cls, qkv, wq, wk1, wk2, wv1, wv2, heads, kv_heads, dim_head, eps):
        assert qkv.is_cuda and qkv.dtype == torch.bfloat16 and qkv.dim() == 3
        assert qkv.shape[-1] == (heads + 4 * kv_heads) * dim_head, 'projection width does not match the head layout'
        if torch.jit.is_tracing():      # (a tracer sees Python Functions only)
            return super().apply(qkv, wq, wk1, wk2, wv1, wv2, heads, kv_heads, dim_head, eps)
        return tuple(_native.torch_ext().qkv_norm(qkv, wq, wk1, wk2, wv1, wv2, heads, kv_heads, dim_head, float(eps)))

    @staticmethod
    def forward(ctx, qkv, wq, wk1, wk2, wv1, wv2, heads, kv_heads, dim_head, eps):
        outs, saved, ctx.sizes = _native.torch_ext().qkv_norm_forward(qkv, wq, wk1, wk2, wv1, wv2, heads, kv_heads, dim_head, float(eps))
        ctx.save_for_backward(*saved)
        return tuple(outs)

    @staticmethod
    def backward(ctx, *grads):
        return (*_native.torch_ext().qkv_norm_backward(ctx.saved_tensors, ctx.sizes, grads), None, None, None, None)


def fused_qkv_norm(qkv, norms, heads, kv_heads, dim_head):
    """``norms``: the five RMSNorm modules in the order q, k1, k2, v1, v2."""
    # eps=None: torch's rms_norm normalises bf16 input in fp32 with the fp32 machine epsilon
    eps = norms[0].eps if norms[0].eps is not None else torch.finfo(torch.float32).eps
    weights = [n.weight if n.elementwise_affine else None for n in norms]
    return FusedQKVNorm.apply(qkv, *weights, heads, kv_heads, dim_head, eps)
