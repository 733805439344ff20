"""The fp32 linear kernels (three-term bf16 splits on the bf16 matrix cores)
against float64, at the edges of each form's tiles, and the non-finite results
they recompute from the fp32 operands."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

SHAPES = [
    # 32 x 32 tiles, K split over four or eight wavefronts (some without a k-step).
    (1, 4, 32), (31, 36, 64), (33, 32, 96), (129, 132, 224),
    # 64 x 64 tiles, ragged both ways.
    (2047, 516, 544), (2049, 1540, 512),
    # 128 x 128 tiles: whole, ragged, several tiles per workgroup, one stage.
    (4096, 1024, 1024), (3999, 1000, 1024), (16385, 1160, 96), (32768, 1024, 32),
]


def _inputs(rows, out_features, in_features, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(rows, in_features, device="cuda", generator=g)
    w = torch.randn(out_features, in_features, device="cuda", generator=g) * in_features ** -0.5
    b = torch.randn(out_features, device="cuda", generator=g)
    return x, w, b


@pytest.mark.parametrize("rows,out_features,in_features", SHAPES)
@pytest.mark.parametrize("bias", [True, False], ids=["bias", "nobias"])
def test_linear_f32_against_float64(gpu_ready, rows, out_features, in_features, bias):
    from transformer_opt.kernels import gelu
    from transformer_opt.kernels.linear_f32 import linear_f32, split_weight

    x, w, b = _inputs(rows, out_features, in_features, rows + in_features)
    b = b if bias else None
    with torch.inference_mode():
        split = split_weight(w)
        y = linear_f32(x, w, split, b)
        exact = torch.matmul(x.double(), w.double().t().contiguous())
        scale = torch.matmul(x.double().abs(), w.double().abs().t().contiguous())
        if bias:
            exact, scale = exact + b.double(), scale + b.double().abs()
        err = (y.double() - exact).abs()
        # Products left out: 2^-24 of |x||w|; two roundings per 16 values
        # of K and sum, and a few at the end.
        assert bool((err <= (2.0 * in_features / 16 + 24) * 2.0 ** -24 * scale).all())
        # No less accurate than the library's fp32 GEMM (2-norm).
        library = F.linear(x, w, b).double() - exact
        assert (y.double() - exact).norm() <= max(library.norm(), 1e-7 * exact.norm())
        z = linear_f32(x, w, split, b, gelu=True)
        torch.testing.assert_close(z, gelu(y), rtol=1e-6, atol=1e-7)
        # The same call gives the same bits.
        assert torch.equal(linear_f32(x, w, split, b), y)


@pytest.mark.parametrize("rows,out_features,in_features", SHAPES + [
    (16, 1024, 4096), (8192, 768, 256), (1000, 516, 544), (700, 1540, 512), (300, 1020, 288)])
@pytest.mark.parametrize("gelu", [False, True], ids=["linear", "gelu"])
def test_terms_made_by_the_call(gpu_ready, rows, out_features, in_features, gelu):
    # Small products split W in registers, the tiled kernel reads terms made
    # beforehand: the same terms, so the same bits where both take one form.
    from transformer_opt.kernels import gelu as exact_gelu
    from transformer_opt.kernels.linear_f32 import linear_f32, split_weight

    x, w, b = _inputs(rows, out_features, in_features, rows + out_features)
    with torch.inference_mode():
        split = split_weight(w)
        y = linear_f32(x, w, None, b, gelu=gelu)
        exact = torch.addmm(b.double(), x.double(), w.double().t().contiguous())
        scale = torch.matmul(x.double().abs(), w.double().abs().t().contiguous()) + b.double().abs()
        bound = (2.0 * in_features / 16 + 24) * 2.0 ** -24 * scale
        given = linear_f32(x, w, split, b, gelu=gelu)
        if not gelu:
            assert bool(((y.double() - exact).abs() <= bound).all())
            assert bool(((y - given).double().abs() <= 2 * bound).all())
        else:
            torch.testing.assert_close(y, exact_gelu(linear_f32(x, w, None, b)), rtol=1e-6, atol=1e-7)
        if in_features <= 96 or rows >= 32768:
            assert torch.equal(y, given)
        # Following the weight: no terms are left over.  (The same bound: the
        # matrix core's sums are not the same bits with every sign turned.)
        w.mul_(-1.0)
        again = linear_f32(x, w, None, -b)
        assert bool(((again.double() + exact).abs() <= bound).all())


@pytest.mark.parametrize("rows,out_features,in_features", [
    (1, 4, 1024), (16, 2048, 8192), (33, 100, 2080), (64, 1020, 4000), (31, 260, 1056), (128, 2048, 8192), (65, 516, 5152)])
@pytest.mark.parametrize("bias", [True, False], ids=["bias", "nobias"])
def test_workgroups_that_share_a_tile(gpu_ready, rows, out_features, in_features, bias):
    # Few tiles of long K, in 32 x 32 and 64 x 64 tiles, k-steps that do not
    # divide among the wavefronts; the workspace holds NaN before the call.
    from transformer_opt import _native
    from transformer_opt.kernels import gelu
    from transformer_opt.kernels.linear_f32 import linear_f32

    need = _native.load().ttk_linear_f32_workspace_size(rows, out_features, in_features)
    tiles = -(-rows // 32) * -(-out_features // 32)
    assert 0 < need != _native.load().ttk_linear_f32_split_bytes(out_features, in_features) and need % 4096 == 0
    assert need >= 2 * 4096 * min(tiles, 256)
    x, w, b = _inputs(rows, out_features, in_features, rows + out_features)
    b = b if bias else None
    x[0, 3] = float("inf")
    if rows > 2:
        x[1] *= 2.0 ** -118
        x[2] = 0.0
    with torch.inference_mode():
        junk = torch.full((need // 4,), float("nan"), device="cuda")
        del junk
        y = linear_f32(x, w, None, b)
        assert torch.equal(linear_f32(x, w, None, b).nan_to_num(1.0), y.nan_to_num(1.0))
        z = linear_f32(x, w, None, b, gelu=True)
        torch.testing.assert_close(z, gelu(y), rtol=1e-6, atol=1e-7, equal_nan=True)
        exact = torch.matmul(x.double(), w.double().t().contiguous())
        scale = torch.matmul(x.double().abs(), w.double().abs().t().contiguous())
        if bias:
            exact, scale = exact + b.double(), scale + b.double().abs()
    assert torch.equal(y[0].double(), exact[0])  # infinities of either sign
    # Row 1 is a plain fp32 sum: K roundings, and the spacing of subnormal numbers.
    bound = (2.0 * in_features / 16 + 24) * 2.0 ** -24 * scale
    bound[1:2] = (in_features / 2 + 2) * 2.0 ** -24 * scale[1:2] + in_features * 2.0 ** -149
    assert bool(((y.double() - exact).abs() <= bound)[1:].all())


@pytest.mark.parametrize("rows,out_features,in_features", [(128, 256, 64), (2048, 512, 512), (8192, 4096, 1024)])
def test_a_single_product_is_rounded_about_once(gpu_ready, rows, out_features, in_features):
    # Rows with one nonzero value: 2^-24 of the product left out, 2^-24 in the
    # last addition, and the small products' own roundings (2^-8 of that each).
    from transformer_opt.kernels.linear_f32 import linear_f32, split_weight

    x, w, _ = _inputs(rows, out_features, in_features, 11)
    at = torch.arange(rows, device="cuda")
    one = torch.zeros_like(x)
    one[at, at % in_features] = x[at, at % in_features]
    with torch.inference_mode():
        y = linear_f32(one, w, split_weight(w), None).double()
        exact = torch.matmul(one.double(), w.double().t().contiguous())
    assert bool(((y - exact).abs() <= (2.0 + 2.0 ** -5) * 2.0 ** -24 * exact.abs()).all())


@pytest.mark.parametrize("exponent", [-90, -118, -124])
@pytest.mark.parametrize("rows,out_features,in_features", [(40, 64, 64), (2048, 512, 512), (4096, 1024, 1024)])
def test_operands_below_the_range_of_three_terms(gpu_ready, rows, out_features, in_features, exponent):
    # Below 2^-110 a value loses bits as three bf16 terms: rows of such values
    # (the others stay ordinary) and weights, the results plain fp32's.
    from transformer_opt.kernels.linear_f32 import linear_f32, split_weight

    x, w, _ = _inputs(rows, out_features, in_features, 17)
    x[::3] *= 2.0 ** exponent
    w[1::5] *= 2.0 ** -20
    x[1] = 0.0
    for a, b in ((x, w), (x[2::3].contiguous(), w * 2.0 ** exponent)):
        with torch.inference_mode():
            y = linear_f32(a, b, split_weight(b), None).double()
            exact = torch.matmul(a.double(), b.double().t().contiguous())
            scale = torch.matmul(a.double().abs(), b.double().abs().t().contiguous())
        # A sum of K rounded products, and the spacing of subnormal numbers.
        bound = (in_features / 2 + 2) * 2.0 ** -24 * scale + in_features * 2.0 ** -149
        assert bool(((y - exact).abs() <= bound).all())


@pytest.mark.parametrize("rows,out_features,in_features", [(40, 64, 64), (2048, 512, 512), (4096, 1024, 1024)])
def test_non_finite_results_are_those_of_the_fp32_operands(gpu_ready, rows, out_features, in_features):
    from transformer_opt.kernels.linear_f32 import linear_f32, split_weight

    x, w, b = _inputs(rows, out_features, in_features, 3)
    inf = float("inf")
    x[3, 5], x[7, 1], x[9, 0], x[11, 2] = inf, float("nan"), 3.4e38, -inf
    w[4] = 1.0        # +inf, NaN, an overflow past bf16 and -inf meet a plain row
    w[6, 5] = 0.0     # 0 * inf
    w[8, 3] = inf
    x[:, 3] = x[:, 3].abs() + 1.0
    x[9, 1:] = 0.0
    with torch.inference_mode():
        y = linear_f32(x, w, split_weight(w), b)
        exact = torch.addmm(b.double(), x.double(), w.double().t().contiguous()).float()
    assert torch.equal(torch.isnan(y), torch.isnan(exact))
    at_inf = torch.isinf(exact)
    assert bool(at_inf.any()) and torch.equal(y[at_inf], exact[at_inf])
    fine = torch.isfinite(exact)
    torch.testing.assert_close(y[fine], exact[fine], rtol=1e-5, atol=1e-4)


def test_split_weight_declines_what_the_kernel_cannot_take(gpu_ready):
    from transformer_opt.kernels.linear_f32 import linear_f32_supported, split_weight

    ok = torch.zeros(64, 64, device="cuda")
    assert split_weight(ok).numel() == 64 * 64 * 6
    for bad in (ok.cpu(), ok.bfloat16(), ok.t()[:, :33], ok[:, :48], ok[:62], ok.view(-1)):
        assert split_weight(bad) is None
    x = torch.zeros(5, 64, device="cuda")
    assert linear_f32_supported(x, ok, None)
    assert not linear_f32_supported(x[:, :32], ok, None)
    assert not linear_f32_supported(x.double(), ok, None)
    with torch.enable_grad():
        assert not linear_f32_supported(x.clone().requires_grad_(), ok, None)
        assert not linear_f32_supported(x, ok.clone().requires_grad_(), None)
    with torch.autocast("cuda"):
        assert not linear_f32_supported(x, ok, None)


def test_terms_that_are_not_the_weights_are_refused(gpu_ready):
    from transformer_opt.kernels.linear_f32 import linear_f32, split_weight

    x, w = torch.zeros(5, 64, device="cuda"), torch.zeros(64, 64, device="cuda")
    split = split_weight(w)
    smaller, larger = split_weight(w[:32]), split_weight(torch.zeros(68, 64, device="cuda"))
    for bad in (smaller, larger, split.cpu(), split.view(torch.float32), split[::2], split[16:], w):
        with pytest.raises(ValueError, match="split"):
            linear_f32(x, w, bad, None)
    for weight in (w.t(), w.bfloat16(), w.double(), w.cpu(), w[0]):
        with pytest.raises(ValueError, match="unsupported"):
            linear_f32(x, weight, split, None)
    assert torch.equal(linear_f32(x, w, split, None), torch.zeros_like(x))


def _model(execution_mode, layers=2):
    from transformer_opt.submission import TransformerConfig, UserOptimizedTransformer

    torch.manual_seed(5)
    model = UserOptimizedTransformer(TransformerConfig(2, 96, 128, 4, 256, layers, True),
                                     execution_mode=execution_mode)
    return model.cuda().eval()


def _fresh(model, x):
    """What a model that never saw other weights gives."""
    fresh = _model("eager")
    fresh.load_state_dict(model.state_dict())
    with torch.inference_mode():
        return fresh(x)


def test_edited_weights_are_seen_on_every_stream(gpu_ready):
    # In-place edits, eager calls on the editing stream and on one ordered
    # after it.
    model = _model("eager")
    x = torch.randn(2, 96, 128, device="cuda")
    side = torch.cuda.Stream()
    with torch.inference_mode():
        first = model(x).clone()
    with torch.no_grad():
        model.layers[0].ffn_out.weight.mul_(-1.0)
        model.layers[1].attention.k_proj.weight.mul_(0.5)
    expected = _fresh(model, x)
    with torch.inference_mode():
        edited = model(x).clone()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            again = model(x)
        torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(edited, expected) and torch.equal(again, expected)
    assert not torch.allclose(first, expected)


@pytest.mark.parametrize("execution_mode", ["eager", "auto"])
@pytest.mark.parametrize("name", ["attention.out_proj", "ffn_in", "ffn_out"])
def test_writes_that_leave_no_trace_reach_the_projections(gpu_ready, execution_mode, name):
    # ``.data`` writes change neither the parameter's identity nor its
    # version: eager calls and replays read the parameter itself.
    model = _model(execution_mode)
    x = torch.randn(2, 96, 128, device="cuda")
    weight = model.get_submodule(f"layers.0.{name}").weight
    with torch.inference_mode():
        before = model(x).clone()
        weight.data.copy_(weight.data.flip(0) * 1.5)
        after = model(x).clone()
    assert not torch.allclose(before, after)
    assert torch.equal(after, _fresh(model, x))


def test_a_callers_graph_follows_in_place_edits(gpu_ready):
    # The caller's own capture after a warm-up: it reads the parameters
    # themselves and memory that lives as long as the graph.
    model = _model("eager")
    x = torch.randn(2, 96, 128, device="cuda")
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.inference_mode(False), torch.no_grad():
        with torch.cuda.stream(side):
            model(x)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = model(x)
        for scale in (-1.0, 0.5, 3.0):
            model.layers[0].ffn_in.weight.mul_(scale)
            model.layers[1].ffn_out.weight.mul_(scale)
            model.layers[1].attention.out_proj.weight.mul_(scale)
            eager = model(x)
            # Whatever an edit let go of is somebody else's memory by now.
            junk = [torch.full((n,), float("nan"), device="cuda") for n in (1 << 12, 1 << 14, 1 << 16, 1 << 18)]
            graph.replay()
            assert torch.equal(out, eager) and torch.equal(eager, _fresh(model, x))
            del junk
