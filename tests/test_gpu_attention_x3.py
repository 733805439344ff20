"""The fp32 attention kernel that runs on the bf16 matrix cores (head dims 32,
64, 128): accuracy against float64 at the edges of its tiles, overlapping and
strided rows, and operands its three-term splits cannot carry."""

from __future__ import annotations

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _exact(q, k, v, mask, causal, scale):
    """float64 attention (rows without an allowed key: zeros) and, per output,
    sum_t P |v|."""
    qh, kt, vh = (t.double().permute(p).contiguous() for t, p in ((q, (0, 2, 1, 3)), (k, (0, 2, 3, 1)), (v, (0, 2, 1, 3))))
    s = torch.matmul(qh, kt) * scale
    seq = q.shape[1]
    if causal:
        s = s.masked_fill(torch.ones(seq, seq, dtype=torch.bool, device=q.device).triu(1), -math.inf)
    if mask is not None:
        s = s.masked_fill(~mask[:, None, None, :], -math.inf)
    weights = torch.softmax(s, -1)
    weights = torch.where(torch.isneginf(s.amax(-1, keepdim=True)), torch.zeros_like(weights), weights)
    back = (0, 2, 1, 3)
    return torch.matmul(weights, vh).permute(back), torch.matmul(weights, vh.abs()).permute(back)


@pytest.mark.parametrize("seq_len", [1, 31, 32, 33, 64, 95, 96, 97, 129, 255, 257, 700])
@pytest.mark.parametrize("head_dim", [32, 64, 128])
@pytest.mark.parametrize("causal", [False, True], ids=["noncausal", "causal"])
@pytest.mark.parametrize("masked", [False, True], ids=["nomask", "masked"])
def test_error_against_float64(gpu_ready, seq_len, head_dim, causal, masked):
    from transformer_opt.kernels import hip_attention

    g = torch.Generator(device="cuda").manual_seed(seq_len * head_dim)
    packed = torch.randn(2, seq_len, 3, 3, head_dim, device="cuda", generator=g)
    q, k, v = packed.unbind(2)
    mask = torch.rand(2, seq_len, device="cuda", generator=g) < 0.7 if masked else None
    with torch.inference_mode():
        out = hip_attention(q, k, v, mask, causal=causal)
        exact, spread = _exact(q, k, v, mask, causal, head_dim ** -0.5)
    # fp32 scores up to ~6 in magnitude (8 in exp2 units): their rounding and
    # the exponential's move a weight by about 8 * 2^-23; sums over the keys
    # and the division add a few 2^-24 each.
    bound = (8 + 4 + seq_len / 32) * 2.0 ** -23 * spread + 1e-30
    assert bool(((out.double() - exact).abs() <= bound).all())


@pytest.mark.parametrize("seq_len", [1, 32, 33, 64])
@pytest.mark.parametrize("head_dim,batch", [(128, 87), (128, 261), (64, 515), (32, 175), (32, 343)])
@pytest.mark.parametrize("causal", [False, True], ids=["noncausal", "causal"])
@pytest.mark.parametrize("masked", [False, True], ids=["nomask", "masked"])
def test_heads_that_share_a_workgroup(gpu_ready, seq_len, head_dim, batch, causal, masked):
    # Up to 64 keys and more heads than workgroup slots (256, or 512 below head
    # dim 128): one (head dim 32 up to 768 heads) to four a workgroup, the last
    # one with fewer.
    # Non-finite operands of a head stay in it.
    from transformer_opt.kernels import hip_attention

    g = torch.Generator(device="cuda").manual_seed(seq_len * head_dim + batch)
    packed = torch.randn(batch, seq_len, 3, 3, head_dim, device="cuda", generator=g)
    q, k, v = packed.unbind(2)
    mask = None
    if masked:
        mask = torch.rand(batch, seq_len, device="cuda", generator=g) < 0.7
        mask[:, 0] = True
        mask[3] = False
    with torch.inference_mode():
        clean = hip_attention(q, k, v, mask, causal=causal)
        exact, spread = _exact(q, k, v, mask, causal, head_dim ** -0.5)
    bound = (8 + 4 + seq_len / 32) * 2.0 ** -23 * spread + 1e-30  # as above
    assert bool(((clean.double() - exact).abs() <= bound).all())
    v[5, 0, 1, 3], k[9, 0, 2, 1], v[batch - 1, 0, 2, 0] = math.inf, math.nan, -math.inf
    with torch.inference_mode():
        out = hip_attention(q, k, v, mask, causal=causal)
    out = out.clone()
    assert not bool(out[5, :, 1, 3].isfinite().any()) and bool(out[9, :, 2].isnan().all())
    assert not bool(out[batch - 1, :, 2, 0].isfinite().any())
    for at in ((5, 1), (9, 2), (batch - 1, 2)):
        out[at[0], :, at[1]] = clean[at[0], :, at[1]]
    assert torch.equal(out, clean) or bool(((out.double() - exact).abs() <= bound).all())


@pytest.mark.parametrize("seq_len", [128, 1024])
@pytest.mark.parametrize("head_dim", [32, 64, 128])
def test_no_pull_towards_zero(gpu_ready, seq_len, head_dim):
    # All products of P.V positive: what is left out of them has either sign,
    # so the mean error stays below half a unit in the last place (2^-24).
    from transformer_opt.kernels import hip_attention

    g = torch.Generator(device="cuda").manual_seed(head_dim)
    q, k, v = (torch.randn(4, seq_len, 4, head_dim, device="cuda", generator=g) for _ in range(3))
    v = v.abs() + 0.5
    with torch.inference_mode():
        out = hip_attention(q, k, v, causal=False)
        exact, _ = _exact(q, k, v, None, False, head_dim ** -0.5)
    assert abs((out.double() / exact - 1.0).mean().item()) <= 2.0 ** -24


@pytest.mark.parametrize("head_dim", [32, 64, 128])
def test_scores_of_one_product_are_rounded_about_once(gpu_ready, head_dim):
    # Scores up to 220 in exp2 units from one product each, neighbours close
    # enough to share a row's weight: the error is the score's rounding.  As
    # much of it as products that are rounded once give, 8 % for the 2^-24 of
    # each that is left out, and 2^-24 for the sums.
    from transformer_opt.kernels import hip_attention

    g = torch.Generator(device="cuda").manual_seed(head_dim)
    seq, scale = 512, head_dim ** -0.5
    at = torch.arange(seq, device="cuda").float()[None, :, None]
    got = rounded = 0.0
    for column in range(4):
        q, k = torch.zeros(2, 1, seq, 4, head_dim, device="cuda")
        q[..., column] = 1.0 + 0.1 * torch.rand(1, seq, 4, device="cuda", generator=g)
        k[..., column] = 0.3 / scale * at * (1.0 + 1e-3 * torch.rand(1, seq, 4, device="cuda", generator=g))
        v = torch.randn(1, seq, 4, head_dim, device="cuda", generator=g)
        with torch.inference_mode():
            exact, _ = _exact(q, k, v, None, True, scale)
            out = hip_attention(q, k, v, causal=True)
            s = (q[..., column] * (scale * math.log2(math.e))).permute(0, 2, 1)[..., None] \
                * k[..., column].permute(0, 2, 1)[:, :, None]
            s = s.double().masked_fill(torch.ones(seq, seq, dtype=torch.bool, device="cuda").triu(1), -math.inf)
            weights = torch.softmax(s * math.log(2.0), -1)
            plain = torch.matmul(weights, v.double().permute(0, 2, 1, 3).contiguous()).permute(0, 2, 1, 3)
        got += ((out.double() - exact).norm() / exact.norm()).item()
        rounded += ((plain - exact).norm() / exact.norm()).item()
    print(f"head_dim {head_dim}: {got / 4:.3e}, rounded products {rounded / 4:.3e}")
    assert got <= 1.08 * rounded + 4 * 2.0 ** -24


@pytest.mark.parametrize("exponent", [-90, -118])
@pytest.mark.parametrize("head_dim", [32, 64, 128])
def test_values_below_the_range_of_three_terms(gpu_ready, head_dim, exponent):
    # Values too small for three bf16 terms, and ordinary ones under weights as
    # small (every other value zero): the results of plain fp32 arithmetic.
    from transformer_opt.kernels import hip_attention

    g = torch.Generator(device="cuda").manual_seed(head_dim)
    q, k, v = (torch.randn(2, 150, 3, head_dim, device="cuda", generator=g) for _ in range(3))
    with torch.inference_mode():
        out = hip_attention(q, k, v * 2.0 ** exponent, causal=True).double()
        exact, spread = _exact(q, k, v * 2.0 ** exponent, None, True, head_dim ** -0.5)
    bound = (8 + 4 + 150 / 32) * 2.0 ** -23 * spread + 2.0 ** -146
    assert bool(((out - exact).abs() <= bound).all())
    # Scores in exp2 units: -exponent at key 3, whose value is zero; 0 at the
    # others.
    q, k = torch.zeros(2, 2, 150, 3, head_dim, device="cuda")
    q[..., 0] = 1.0
    k[:, 3, :, 0] = -exponent * math.log(2.0)
    v[:, 3] = 0.0
    with torch.inference_mode():
        out = hip_attention(q, k, v, scale=1.0, causal=False).double()
        exact, spread = _exact(q, k, v, None, False, 1.0)
    # The score is -exponent in magnitude: its rounding moves a weight by 2^-17.
    bound = (2.0 ** -17 + 150 / 2 * 2.0 ** -24) * spread + 2.0 ** -146
    assert bool(((out - exact).abs() <= bound).all())


def test_rows_that_overlap_and_broadcast(gpu_ready):
    from transformer_opt.kernels import hip_attention

    g = torch.Generator(device="cuda").manual_seed(9)
    q = torch.randn(2, 77, 4, 64, device="cuda", generator=g)
    row = torch.randn(2, 1, 4, 64, device="cuda", generator=g)
    line = torch.randn(2, 80 * 16, device="cuda", generator=g)
    window = line.as_strided((2, 77, 4, 64), (80 * 16, 16, 0, 1))  # rows 16 values apart
    with torch.inference_mode():
        for k, v in ((row.expand(2, 77, 4, 64), window), (window, row.expand(2, 77, 4, 64)), (window, window)):
            got = hip_attention(q, k, v, causal=True)
            want = hip_attention(q, k.contiguous(), v.contiguous(), causal=True)
            assert torch.equal(got, want)


@pytest.mark.parametrize("head_dim", [32, 64, 128])
def test_non_finite_operands_give_the_fp32_results(gpu_ready, head_dim):
    # Infinities and NaN in q, k or v, and values that round to infinity in
    # bf16: the same finite rows, infinities and NaN as plain fp32 arithmetic.
    from transformer_opt.kernels import hip_attention

    g = torch.Generator(device="cuda").manual_seed(head_dim)
    q, k, v = (torch.randn(1, 130, 5, head_dim, device="cuda", generator=g) for _ in range(3))
    inf, nan = math.inf, math.nan
    k[0, 40, 0, 3] = inf     # scores of +-inf: a row of NaN, or the key drops out
    q[0, 7, 1, 0] = nan      # one NaN row
    v[0, 0, 2, 5] = -inf     # one output column (key 0: every row weighs it)
    v[0, 0, 3, 2] = 3.4e38   # finite, infinite as bf16
    k[0, 20, 4, :] = 0.0
    k[0, 20, 4, 1] = 3.4e38  # one row's score overflows, the others' do not
    q[0, :, 4, 1] = q[0, :, 4, 1].clamp(-2.0, 2.0)
    q[0, 50, 4, 1] = 1000.0
    scale = head_dim ** -0.5
    with torch.inference_mode():
        out = hip_attention(q, k, v, causal=True, scale=scale)
        s = torch.matmul((q * scale).permute(0, 2, 1, 3).contiguous(), k.permute(0, 2, 3, 1).contiguous()).cpu()
        s = s.masked_fill(torch.ones(130, 130, dtype=torch.bool).triu(1), -inf)
        top = s.masked_fill(s.isnan(), -inf).amax(-1, keepdim=True)
        weights = torch.exp(s - top)
        weights = weights / weights.sum(-1, keepdim=True)
        terms = weights[..., None] * v.permute(0, 2, 1, 3).cpu()[:, :, None]
        want = terms.sum(-2).permute(0, 2, 1, 3)
    out = out.cpu()
    for head in range(5):
        a, b = out[:, :, head], want[:, :, head]
        both = torch.isfinite(a) & torch.isfinite(b)
        torch.testing.assert_close(a[both], b[both], rtol=2e-4, atol=2e-4)
        assert torch.equal(torch.isfinite(a), torch.isfinite(b)), head
