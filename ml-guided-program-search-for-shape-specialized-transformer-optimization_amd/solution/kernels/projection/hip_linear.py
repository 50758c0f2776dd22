"""The small fp32 Linear layers of a model on the gfx950 kernel.

Counterpart of the reference's ``nn.Linear`` projections
(solution/transformer.py:291-353) for fp32 models of few rows: the same
operands and result (``sah_linear_f32``, csrc/linear_f32.hip).  ``project``
takes a call that it is measured faster on and returns None for every other
one, which then runs ``F.linear``.
"""

from __future__ import annotations

import torch
from torch import nn
from torch.autograd import forward_ad

from ..hip._library import (
    SAH_ACTIVATION_GELU_EXACT,
    SAH_ACTIVATION_NONE,
    check_status,
    is_gfx950,
    load_library,
    stream_handle,
)

# One round of the 256 CUs in 32 x 32 tiles, or for a longer K in 16 x 16
# tiles (GPU time in us, library / this kernel):
#   256 x 256 -> 256     63 / 4.7     512 x 256 -> 768     5.8 /  7.8
#   256 x 256 -> 1024   5.6 / 4.9    1024 x 256 -> 1024    8.0 / 13.8
#   100 x 128 -> 128   11.4 / 3.8
#   256 x 512 -> 256    117 / 5.9     256 x 2048 -> 256    7.1 / 10.4
#   256 x 1024 -> 256   5.8 / 6.0     100 x 640 -> 512     4.9 /  6.0
#   16 x 512 -> 512     4.5 / 5.8      16 x 1024 -> 4096   5.8 /  6.5
# Within the rule the library's time is 3.6-172 us, this kernel's 3.1-6.5, at most
# 1.4 us behind.  A call also costs the host about half of F.linear's (10 us less),
# which is what bounds a forward of these sizes; with GELU the elementwise launch
# goes too (256 x 256 -> 1024 8.2 / 5.3).  Replayed from a graph, where the host
# does not count, whole forwards of four layers gain as well (B1 S16: D 256
# 223 / 132 us, D 512 231 / 178, D 1024 280 / 190, with the attention's share).
# (The 16-bit tile kernels were tried here too: at 16384 x 512 -> 1536 and
# 512 -> 512 they are 4-9% faster than the library alone, but the forward of that
# stack measured the same, 835 us.  A program that selects them: B64 S256 D512,
# four layers, 813 us by default, 807 with the Linear + GELU operator, 800 with
# it and the native QKV layout.)
_MAX_TILES = 256
_MAX_IN = 384
_MAX_IN_SMALL_TILES = 1024


def _serves(rows: int, in_features: int, out_features: int, dtype: torch.dtype) -> bool:
    """The rule on sizes and types."""

    return (
        dtype == torch.float32
        and in_features <= _MAX_IN_SMALL_TILES
        and in_features % 128 == 0
        and out_features % 32 == 0
        and (
            (rows + 31) // 32 * (out_features // 32)
            if in_features <= _MAX_IN
            else (rows + 15) // 16 * (out_features // 16)
        )
        <= _MAX_TILES
    )


def _is_plain(module: nn.Linear, value: torch.Tensor) -> bool:
    """Whether calling ``module`` is no more than one F.linear on plain
    tensors: nothing observes, differentiates or casts the call."""

    if torch.is_grad_enabled() or torch.is_autocast_enabled("cuda"):
        return False
    if forward_ad._current_level >= 0:  # dual tensors carry tangents under no_grad too
        return False
    if type(value) is not torch.Tensor:
        return False
    for parameter in (module._parameters["weight"], module._parameters["bias"]):
        if parameter is not None and type(parameter) not in (nn.Parameter, torch.Tensor):
            return False
    if module._forward_hooks or module._forward_pre_hooks or "forward" in module.__dict__:
        return False
    if type(module).forward is not nn.Linear.forward or type(module).__call__ is not nn.Module.__call__:
        return False
    registry = nn.modules.module
    if registry._global_forward_hooks or registry._global_forward_pre_hooks:
        return False
    return not (
        torch._C._len_torch_dispatch_stack()
        or torch._C._len_torch_function_stack()
        or torch._C._functorch.peek_interpreter_stack() is not None
    )


def project(module: nn.Linear, value: torch.Tensor, *, gelu: bool = False) -> torch.Tensor | None:
    """``module(value)``, with ``gelu`` the exact GELU of it, on the gfx950
    kernel, or None where it does not serve the call (size, type, layout, or a
    call that something observes)."""

    # before the sizes, so that a trace holds no guard on them
    if value.dtype is not torch.float32 or torch.compiler.is_compiling() or torch.jit.is_tracing():
        return None
    # as registered: reading a parametrized weight computes it (spectral_norm
    # takes a power iteration each time), which is for the module to do once
    weight, bias = module._parameters.get("weight"), module._parameters.get("bias")
    if weight is None or "bias" not in module._parameters:
        return None
    dtype = value.dtype
    out_features, in_features = weight.shape
    if not value.is_cuda or value.ndim < 2 or value.shape[-1] != in_features:
        return None
    rows = value.numel() // in_features
    if rows == 0 or not _serves(rows, in_features, out_features, dtype) or not _is_plain(module, value):
        return None
    if weight.dtype != dtype or weight.device != value.device or not (value.is_contiguous() and weight.is_contiguous()):
        return None
    pointers = (value.data_ptr(), weight.data_ptr(), 0 if bias is None else bias.data_ptr())
    if (pointers[0] | pointers[1] | pointers[2]) % 16:
        return None
    if bias is not None and (bias.dtype != dtype or bias.device != value.device or not bias.is_contiguous()):
        return None
    if not is_gfx950(value.device):
        return None
    output = torch.empty((*value.shape[:-1], out_features), device=value.device, dtype=dtype)
    status = load_library().sah_linear_f32(
        pointers[0],
        pointers[1],
        pointers[2] or None,
        output.data_ptr(),
        rows,
        in_features,
        out_features,
        in_features,
        out_features,
        SAH_ACTIVATION_GELU_EXACT if gelu else SAH_ACTIVATION_NONE,
        stream_handle(value.device),
    )
    check_status(status, "sah_linear_f32")
    return output


__all__ = ["project"]
