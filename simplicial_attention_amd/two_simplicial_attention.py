"""Sliding-window 2-simplicial attention on MI355X: autograd Function, functional
wrapper and multi-head module.

Same names, argument order, tensor layouts and defaults as
simplicial_attention/triton_two_simplicial_attention.py of the reference
(Function :718-1008, wrapper :1020-1056, module :1062-1081); the device work is done
by hand-written gfx950 kernels reached through the C ABI of libsa2.so.
"""
from __future__ import annotations

import os
import threading

from functools import partial

import torch
import torch.nn.functional as F
from torch import Tensor
from torch.autograd import Function

from . import _native
from .simplicial_mha import HigherOrderAttention


def save_partials_max_bytes() -> int:
    """Largest per-call buffer of saved value partials the forward may allocate for the
    backward (bytes).  ``SA2_SAVE_PARTIALS_MAX_GIB`` overrides the default of 16 GiB;
    0 switches the saving off (the backward then recomputes, as the reference does)."""
    return int(float(os.environ.get('SA2_SAVE_PARTIALS_MAX_GIB', '16')) * (1 << 30))


def save_partials_total_fraction() -> float:
    """Share of a device's memory that all live saved partials together may occupy
    (``SA2_SAVE_PARTIALS_TOTAL_FRACTION``, default 0.25)."""
    return float(os.environ.get('SA2_SAVE_PARTIALS_TOTAL_FRACTION', '0.25'))


class _PartialsBudget:
    """Bytes of saved value partials alive per device (between a forward and the end of its
    backward).  The partials are ``w2`` times the size of ``q`` per call, so a deep model
    would otherwise keep ``layers * w2`` activations where the reference keeps ``layers``:
    a call saves them only while (a) the call's buffer fits the per-call cap and (b) all live
    buffers together stay below a fraction of the device's total memory.  Otherwise the
    backward recomputes, as the reference does, at about 20 % more time per layer.  The rule
    looks at sizes only, never at how much memory happens to be free: the two backward paths
    differ in the last bf16 digit of dV2, and a model's gradients must not depend on what
    else the allocator holds."""

    def __init__(self, released=lambda index: 0):
        self.live = {}
        self.total = {}
        self.released = released        # bytes of buffers that have died since the process began, per device
        self.lock = threading.Lock()

    def admit(self, nbytes: int, device, total_memory=None) -> bool:
        if nbytes <= 0 or nbytes > save_partials_max_bytes():
            return False
        index = device if isinstance(device, int) else torch.device(device).index
        index = torch.cuda.current_device() if index is None else index
        with self.lock:
            if total_memory is None:
                if index not in self.total:
                    self.total[index] = torch.cuda.get_device_properties(index).total_memory
                total_memory = self.total[index]
            live = self.live.get(index, 0)
            if live - self.released(index) + nbytes > save_partials_total_fraction() * total_memory:
                return False
            self.live[index] = live + nbytes
        return True

    def release(self, nbytes: int, index: int) -> None:
        with self.lock:
            self.live[index] = max(self.live.get(index, 0) - nbytes, 0)


# (the native host path allocates the buffers and counts the bytes of those that die)
partials_budget = _PartialsBudget(lambda index: _native.torch_ext().released_bytes(index))


class SlidingTwoSimplicialAttention(Function):
    """``apply(q, k1, k2, v1, v2, w1, w2, causal[, scale]) -> out``; every tensor ``(b, n, h, d)``.

    ``k1, k2, v1, v2`` may carry fewer heads than ``q`` (grouped queries, query head
    ``h`` reads key/value head ``h // groups``); the reference's Function receives
    them already repeated, which is the special case of one group per head.
    Gradients come back in the order ``dq, dk1, dk2, dv1, dv2`` in the input dtype.
    ``scale`` (not an argument of the reference's Function, which always uses
    ``dim_head ** -0.5``) overrides the softmax scale; the functional wrapper passes it
    when it has zero-padded the head dimension.
    """

    @classmethod
    def apply(cls, q, k1, k2, v1, v2, w1, w2, causal, scale=None):
        # The kernels compute on bf16 operands with fp32 accumulation, as the reference's do for any input dtype
        # (triton_two_simplicial_attention.py:110-112, 150-152); other dtypes are cast on the way in and results
        # returned in the caller's dtype.  Checks, allocation, launches and the autograd node are native
        # (csrc/sa2_torch.cpp): from here they cost more than the kernels of a small call.
        if not causal:
            raise NotImplementedError('only causal=True is defined for the sliding windows')
        # A tracer (torch.jit.trace) sees Python Functions only: it gets this one.
        if torch.jit.is_tracing():
            return super().apply(q, k1, k2, v1, v2, w1, w2, causal, scale)
        return _native.torch_ext().attend(q, k1, k2, v1, v2, int(w1), int(w2), scale, False, partials_budget.admit)

    @staticmethod
    def forward(ctx, q, k1, k2, v1, v2, w1, w2, causal, scale=None):
        if not causal:
            raise NotImplementedError('only causal=True is defined for the sliding windows')
        out, saved, ctx.sizes, ctx.scale = _native.torch_ext().attend_forward(
            q, k1, k2, v1, v2, int(w1), int(w2), scale, any(ctx.needs_input_grad[:5]), partials_budget.admit)
        ctx.save_for_backward(*saved)
        return out

    @staticmethod
    def backward(ctx, dout):
        return (*_native.torch_ext().attend_backward(ctx.saved_tensors, ctx.sizes, ctx.scale, dout), None, None, None, None)


_sliding_two_simplicial_attn = SlidingTwoSimplicialAttention.apply
_DTYPES = (torch.bfloat16, torch.float16, torch.float32)


def sliding_two_simplicial_attn(
    q: Tensor,                      # (b, n, hq, d)
    keys: tuple[Tensor, Tensor],    # (b, n, h, d) * 2
    values: tuple[Tensor, Tensor],  # (b, n, h, d) * 2
    w1=512,
    w2=32,
    causal=True,
    pad_to_multiple_of=64,
):
    """Functional entry point, signature of triton_two_simplicial_attention.py:1020-1056.

    Grouped-query heads are resolved by index arithmetic inside the kernels and a
    ragged sequence end is masked there, so nothing is repeated or padded here;
    ``pad_to_multiple_of`` is accepted for compatibility and has no effect on the
    result (zero rows appended after a causal sequence cannot influence it).

    Beyond the reference (whose kernels are written for bf16 and a head dimension of
    64): float16 and float32 tensors are computed in bfloat16 and the result returned
    in the input dtype; any head dimension up to 256, and a value head dimension
    different from the query/key one, are zero-padded to the kernels' 32, 64, 128 or 256
    (padded query/key channels add nothing to the logits, padded value channels give
    zero outputs that are sliced off; the softmax scale stays that of the true
    query/key dimension).
    """
    if len(keys) != 2 or len(values) != 2:
        raise AssertionError('two key sets and two value sets are required')
    q_heads, k_heads = q.shape[-2], keys[0].shape[-2]
    assert q_heads % k_heads == 0, 'query heads must be a multiple of key/value heads'
    (k1, k2), (v1, v2) = keys, values
    dtype, dim_qk, dim_v = q.dtype, q.shape[-1], v1.shape[-1]
    if dtype not in _DTYPES:
        raise TypeError(f'unsupported dtype {dtype}')
    if k1.shape[-1] != dim_qk or k2.shape[-1] != dim_qk or v2.shape[-1] != dim_v:
        raise ValueError('q, k1, k2 must share one head dimension and v1, v2 another')
    dim = max(dim_qk, dim_v)
    if dim > 256:
        raise NotImplementedError(f'head dimension {dim} is not covered by the kernels (at most 256)')
    if dtype is torch.bfloat16 and dim_qk == dim_v and dim in (32, 64, 128, 256):
        return _sliding_two_simplicial_attn(q, k1, k2, v1, v2, w1, w2, causal)
    if not causal:
        raise NotImplementedError('only causal=True is defined for the sliding windows')
    if torch.jit.is_tracing():
        kernel_dim = next(d for d in (32, 64, 128, 256) if dim <= d)
        rows = [F.pad(t.to(torch.bfloat16), (0, kernel_dim - t.shape[-1])) for t in (q, k1, k2, v1, v2)]
        return _sliding_two_simplicial_attn(*rows, w1, w2, causal, dim_qk ** -0.5)[..., :dim_v].to(dtype)
    k1, k2, v1, v2 = (t if t.dtype in _DTYPES else t.to(torch.bfloat16) for t in (k1, k2, v1, v2))
    return _native.torch_ext().attend(q, k1, k2, v1, v2, int(w1), int(w2), None, True, partials_budget.admit)


class SlidingWindowTwoSimplicialMHA(HigherOrderAttention):
    """Multi-head module, constructor of triton_two_simplicial_attention.py:1062-1081."""

    def __init__(self, *args, w1=512, w2=32, **kwargs):
        assert 'number_key_value_sets' not in kwargs
        assert 'head_first_dim' not in kwargs
        attend = partial(sliding_two_simplicial_attn, w1=w1, w2=w2, causal=True)
        super().__init__(*args, number_key_value_sets=2, head_first_dim=False, attend=attend, **kwargs)
