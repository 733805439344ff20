"""fp32 linear layer (optionally with the exact GELU) on the gfx950 HIP kernel.

``linear_f32(x, weight, None, bias, gelu=...)`` returns ``F.linear(x, weight,
bias)``, or its exact GELU, of fp32 tensors: the projections of the fp32
encoder (reference transformer_opt/submission.py:484-508).  The products run on
the bf16 matrix cores, each operand as three bf16 terms that sum to it
(``ttk_linear_f32_fwd_ws``): what is left out of a product is at most 2^-24 of
it, and dense sums come out closer to float64 than an fp32 GEMM's.

Nothing is kept between calls: the weight's terms, where the product is large
enough to want them, are made by each call.  A caller whose weight does not
change may make them once, ``split_weight(weight)``, and pass them instead of
None; it owes a new split after every change of the weight.

The encoder model uses it (``submission.UserOptimizedTransformer``); where
``linear_f32_supported`` declines, the model's library route runs.
"""

from __future__ import annotations

from typing import Optional

import torch

from .. import _native
from .._launch import launch, query


def _float_rows(t: torch.Tensor) -> bool:
    return t.is_cuda and t.dtype == torch.float32 and t.is_contiguous() and t.data_ptr() % 16 == 0


def _weight_taken(weight: torch.Tensor) -> bool:
    """A contiguous fp32 ROCm matrix [N, K] with K a multiple of 32 and N of 4."""
    if weight.ndim != 2 or not _float_rows(weight):
        return False
    n, k = weight.shape
    return n > 0 and k > 0 and n % 4 == 0 and k % 32 == 0 and max(n, k) < 1 << 22


def split_weight(weight: torch.Tensor) -> Optional[torch.Tensor]:
    """The three bf16 terms of ``weight`` [N, K] (N * K * 6 bytes, N rounded up
    to 32), or None when the kernel cannot take the weight."""
    if not _weight_taken(weight):
        return None
    n, k = weight.shape
    lib = _native.load()
    split = torch.empty(lib.ttk_linear_f32_split_bytes(n, k), dtype=torch.uint8, device=weight.device)
    status = launch(weight.get_device(), lib.ttk_linear_f32_split_weight, weight.data_ptr(), split.data_ptr(), n, k, k)
    _native.check(status, "split weight")
    return split


def linear_f32_supported(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor]) -> bool:
    """Whether ``linear_f32`` takes this call.  Calls that autograd or autocast
    would see stay with the library route."""
    if not (_float_rows(x) and _weight_taken(weight)) or x.shape[-1] != weight.shape[1] or x.device != weight.device:
        return False
    if bias is not None and not (_float_rows(bias) and bias.device == x.device):
        return False
    if torch.is_grad_enabled() and (x.requires_grad or weight.requires_grad
                                    or (bias is not None and bias.requires_grad)):
        return False
    return not torch.is_autocast_enabled("cuda") and not torch.compiler.is_compiling()


def linear_f32(x: torch.Tensor, weight: torch.Tensor, split: Optional[torch.Tensor], bias: Optional[torch.Tensor],
               gelu: bool = False) -> torch.Tensor:
    """``F.linear(x, weight, bias)``, with ``gelu`` its exact GELU."""
    if not linear_f32_supported(x, weight, bias):
        raise ValueError("unsupported HIP fp32 linear input")
    lib = _native.load()
    n, k = weight.shape
    y = torch.empty(*x.shape[:-1], n, dtype=x.dtype, device=x.device)
    rows = x.numel() // k
    act = _native.TTK_ACT_GELU if gelu else _native.TTK_ACT_NONE
    index = x.get_device()
    bias_ptr = None if bias is None else bias.data_ptr()
    if split is None:
        nbytes = query(index, lib.ttk_linear_f32_workspace_size, rows, n, k)
        ws = torch.empty(nbytes, dtype=torch.uint8, device=x.device) if nbytes else None
        status = launch(index, lib.ttk_linear_f32_fwd_ws, x.data_ptr(), weight.data_ptr(), bias_ptr, y.data_ptr(),
                        rows, n, k, k, k, n, act, None if ws is None else ws.data_ptr(), nbytes)
    else:
        if (split.device != weight.device or split.dtype != torch.uint8 or not split.is_contiguous()
                or split.numel() != lib.ttk_linear_f32_split_bytes(n, k)):
            raise ValueError("split is not what split_weight gives for a weight of this shape and device")
        status = launch(index, lib.ttk_linear_f32_fwd, x.data_ptr(), weight.data_ptr(), split.data_ptr(), bias_ptr,
                        y.data_ptr(), rows, n, k, k, k, n, act)
    _native.check(status, "fp32 linear")
    return y
