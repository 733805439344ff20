"""Residual + LayerNorm at widths that do not divide into equal lane groups and
on unaligned tensors: a row per lane group, per workgroup, or re-read."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

# fp32 vectors (of 4): 13 and 21 (masked lane groups), 125, 1021 (64 lanes),
# 1025 (workgroup), 4095, 4097 (re-read).  Elements: 33, 1023, 1025 (workgroup),
# 8191, 8193 (re-read).  16-bit vectors hold 8.
WIDTHS = [52, 84, 500, 1000, 4084, 4100, 16380, 16388, 33, 1023, 1025, 4097, 8191, 8193, 32760]


@pytest.mark.parametrize("width", WIDTHS)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("rows,offset", [(1, 0), (7, 0), (67, 0), (9, 1)])
def test_ragged_widths(gpu_ready, width, dtype, rows, offset):
    from transformer_opt.kernels import fused_residual_layer_norm, layer_norm

    g = torch.Generator(device="cuda").manual_seed(width + rows)

    def tensor(*shape):
        # `offset` elements past a 16-byte boundary: the element path.
        n = torch.Size(shape).numel()
        return torch.randn(n + offset, device="cuda", generator=g).to(dtype)[offset:].view(*shape)

    x, u, w, b = tensor(rows, width), tensor(rows, width), tensor(width), tensor(width)
    mask = torch.arange(rows, device="cuda") % 3 != 1
    with torch.inference_mode():
        r, y = fused_residual_layer_norm(x, u, w, b, 1e-5, mask, zero_invalid_residual=True,
                                         zero_invalid_normalized=True)
        plain = layer_norm(x, w, None, 1e-5)
        want_r = (x + u).masked_fill(~mask[:, None], 0)
        want = F.layer_norm(want_r.double(), (width,), w.double(), b.double(), 1e-5).masked_fill(~mask[:, None], 0)
        want_plain = F.layer_norm(x.double(), (width,), w.double(), None, 1e-5)
    assert torch.equal(r, want_r)
    # One rounding of the result (half an ulp), and the statistics': sums of at
    # most 32 values a lane and 8 lane steps, each rounded to fp32.
    ulp = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    for got, exact in ((y, want), (plain, want_plain)):
        bound = ulp * exact.abs() + 48 * 2.0 ** -24 * (exact.abs() + w.double().abs() * 4 + 1) + 1e-7
        assert bool(((got.double() - exact).abs() <= bound).all())


@pytest.mark.parametrize("width", [65, 100, 512, 520, 1001, 1024])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("rows,offset", [(1024, 0), (1025, 0), (1025, 1)])
def test_either_side_of_the_rule_on_rows(gpu_ready, width, dtype, rows, offset):
    test_ragged_widths(gpu_ready, width, dtype, rows, offset)
