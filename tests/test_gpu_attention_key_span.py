"""Key masks whose invalid keys form whole 64-key blocks: attention visits the
span of valid keys only, and its 16-bit kernel drops the mask inside it."""

from __future__ import annotations

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _rows(seq):
    """Masks of every shape the span has to get right, one a row."""
    m = torch.zeros(10, seq, dtype=torch.bool)
    m[0] = True
    m[1, :seq // 2 + 5] = True             # prefix that ends inside a block
    m[2, :128] = True                      # prefix that ends with a block
    m[3, seq - 129:] = True                # left padding
    m[4, 64:192] = True                    # both, on block edges
    m[5, 200:201] = True                   # one key
    m[6, ::3] = True                       # scattered
    m[7] = True
    m[7, 300:301] = False                  # one hole
    m[8, 65:130] = True                    # two valid parts
    m[8, 390:] = True
    return m                               # the last: no valid key


@pytest.mark.parametrize("seq", [512, 513, 577, 640, 1000, 4200])
@pytest.mark.parametrize("head_dim", [8, 32, 64, 128])
@pytest.mark.parametrize("causal", [False, True], ids=["noncausal", "causal"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=["fp32", "bf16", "fp16"])
def test_against_float64(gpu_ready, seq, head_dim, causal, dtype):
    from transformer_opt.kernels import hip_attention

    g = torch.Generator(device="cuda").manual_seed(seq + head_dim)
    mask = _rows(seq).cuda()
    heads = 2 if seq < 4000 else 1
    q, k, v = (torch.randn(len(mask), seq, heads, head_dim, device="cuda", generator=g).to(dtype) for _ in range(3))
    wide = torch.zeros(len(mask), 2 * seq, dtype=torch.bool, device="cuda")
    wide[:, ::2] = mask
    with torch.inference_mode():
        got = hip_attention(q, k, v, mask, causal=causal)
        strided = hip_attention(q, k, v, wide[:, ::2], causal=causal)  # no span: every key visited
        qh, kt, vh = (t.double().permute(p).contiguous() for t, p in ((q, (0, 2, 1, 3)), (k, (0, 2, 3, 1)), (v, (0, 2, 1, 3))))
        s = torch.matmul(qh, kt) * head_dim ** -0.5
        if causal:
            s.masked_fill_(torch.ones(seq, seq, dtype=torch.bool, device="cuda").triu_(1), -math.inf)
        s.masked_fill_(~mask[:, None, None, :], -math.inf)
        weights = torch.softmax(s, -1)
        weights.masked_fill_(torch.isneginf(s.amax(-1, keepdim=True)), 0.0)
        exact = torch.matmul(weights, vh).permute(0, 2, 1, 3)
        spread = torch.matmul(weights, vh.abs()).permute(0, 2, 1, 3)
    # A weight is off by its rounding to the storage type (twice: it also enters
    # the row sum) and by 2^-20 of fp32 scores; the result is rounded once.
    eps = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    bound = (2.5 * eps + (8 + 4 + seq / 32) * 2.0 ** -23) * spread + eps * exact.abs() + 2.0 ** -24
    for name, out in (("span", got), ("strided", strided)):
        assert bool(((out.double() - exact).abs() <= bound).all()), name


@pytest.mark.parametrize("heads", [5, 6, 7, 8, 9, 12], ids=lambda h: f"groups{90 * h}")
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_tile_rule_of_long_masked_launches(gpu_ready, dtype, heads):
    # 90 workgroups a head: up to 512 of them (256 CUs) 64-key tiles, up to 640
    # 32-key tiles, then 64-key ones unless the rows are strided and a round is
    # saved (8 heads: one instead of two; 9: two either way; 12: two instead of
    # three).
    from transformer_opt.kernels import hip_attention

    seq, head_dim = 1100, 128
    g = torch.Generator(device="cuda").manual_seed(heads)
    mask = _rows(seq).cuda()
    q, k, v = (torch.randn(len(mask), seq, heads, head_dim, device="cuda", generator=g).to(dtype) for _ in range(3))
    wide = torch.zeros(len(mask), 2 * seq, dtype=torch.bool, device="cuda")
    wide[:, ::2] = mask
    eps = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]  # the bound of test_against_float64
    with torch.inference_mode():
        outs = {"span": hip_attention(q, k, v, mask), "strided": hip_attention(q, k, v, wide[:, ::2])}
        for b in range(len(mask)):
            qh, kt, vh = (t[b].double().permute(p).contiguous() for t, p in ((q, (1, 0, 2)), (k, (1, 2, 0)), (v, (1, 0, 2))))
            s = torch.matmul(qh, kt).mul_(head_dim ** -0.5).masked_fill_(~mask[b], -math.inf)
            weights = torch.softmax(s, -1) if bool(mask[b].any()) else torch.zeros_like(s)
            exact, spread = torch.matmul(weights, vh), torch.matmul(weights, vh.abs())
            bound = (2.5 * eps + (8 + 4 + seq / 32) * 2.0 ** -23) * spread + eps * exact.abs() + 2.0 ** -24
            for name, out in outs.items():
                assert bool(((out[b].permute(1, 0, 2).double() - exact).abs() <= bound).all()), (name, b)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("value", [math.inf, math.nan])
@pytest.mark.parametrize("row", [3, 600, 767])
def test_non_finite_values_of_dropped_keys(gpu_ready, dtype, value, row):
    # Zero weight times an infinite or NaN value is NaN, also where the key's
    # whole block is invalid; K of an invalid key has no effect.
    from transformer_opt.kernels import hip_attention

    g = torch.Generator(device="cuda").manual_seed(row)
    q, k, v = (torch.randn(1, 768, 2, 64, device="cuda", generator=g).to(dtype) for _ in range(3))
    mask = torch.zeros(1, 768, dtype=torch.bool, device="cuda")
    mask[:, 130:520] = True
    with torch.inference_mode():
        want = hip_attention(q, k, v, mask)
        k[0, row, 0, 5] = value
        assert torch.equal(hip_attention(q, k, v, mask), want)
        v[0, row, 1, 7] = value
        got = hip_attention(q, k, v, mask)
    assert bool(torch.isnan(got[0, :, 1, 7]).all())
    got = torch.where(torch.isnan(got), want, got)
    # Rows with a non-finite sum are computed by other instructions in fp32.
    torch.testing.assert_close(got, want, rtol=1e-2 if dtype != torch.float32 else 1e-5, atol=1e-2 if dtype != torch.float32 else 1e-5)
