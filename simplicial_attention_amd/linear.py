"""Linear layers whose weight gradient runs on this package's kernel where that is the faster one."""
from __future__ import annotations

import torch
import torch.nn.functional as F
from torch import Tensor, nn
from torch.nn.modules import module as _module

from . import _native


# what a call of a linear layer goes through, as torch has it
_FORWARD, _CALL, _CALL_IMPL, _LINEAR = nn.Linear.forward, nn.Linear.__call__, nn.Linear._call_impl, F.linear


def _watched(layer):
    """Someone else sees the calls of this layer, or has changed what it is."""
    if nn.Linear.forward is not _FORWARD or nn.Linear.__call__ is not _CALL or nn.Linear._call_impl is not _CALL_IMPL or F.linear is not _LINEAR:
        return True
    return bool(layer._compiled_call_impl is not None or layer._forward_hooks or layer._forward_pre_hooks or layer._backward_hooks or layer._backward_pre_hooks
                or _module._global_forward_hooks or _module._global_forward_pre_hooks or _module._global_backward_hooks
                or _module._global_backward_pre_hooks or 'forward' in layer.__dict__)


def _faster(rows, out_features, in_features):
    # Measured against the library (us, ours and the library's): 8192 rows, 2048 x 512: 37, 55; 512 x 512: 24, 52; 2048 x 1024: 54, 68;
    # 16384 rows, 2048 x 512: 53, 104; 65536 rows, 2048 x 1024: 308, 368.  The library does not split the rows: with fewer of them
    # (4096 rows, 2048 x 1024: 38, 37) or larger results (65536 rows, 3072 x 1024: 578, 477) it is as fast or faster.
    return rows >= 8192 and out_features % 128 == 0 and in_features % 128 == 0 and out_features * in_features <= 2048 * 1024


def apply_linear(layer, x):
    """``layer(x)``; plain bf16 ``nn.Linear`` layers under training take the node with the kernel of their own."""
    # (torch.fx hands over proxies: the type comes first)
    if (type(x) is not Tensor or type(layer) is not nn.Linear or torch.compiler.is_compiling() or torch.jit.is_tracing()
            or not x.is_cuda or not torch.is_grad_enabled()):
        return layer(x)
    weight, bias = layer.weight, layer.bias
    if (type(weight) is not nn.Parameter or type(bias) not in (nn.Parameter, type(None))
            or x.dtype is not torch.bfloat16 or weight.dtype is not torch.bfloat16 or (bias is not None and bias.dtype is not torch.bfloat16)
            or x.device != weight.device or x.dim() < 2 or x.shape[-1] != weight.shape[1]
            or not _faster(x.numel() // x.shape[-1] if x.shape[-1] else 0, *weight.shape)
            or torch.is_autocast_enabled() or torch._C._len_torch_dispatch_stack() or torch._C._len_torch_function_stack() or _watched(layer)):
        return layer(x)
    return _native.torch_ext().linear(x, weight, bias)
