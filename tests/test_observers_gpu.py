"""Callers that a whole-layer native call must not hide its operators from: transforms, tensor subclasses, autograd."""
import pytest
import torch

pytestmark = pytest.mark.gpu

FP8 = torch.float8_e4m3fn
M, N, K = 6, 384, 256


@pytest.fixture(scope="module")
def linears(dev):
    """name -> f(x, bias): every linear layer that has a whole-layer call."""
    from sglang_amd.quantization import fp8_utils as fu
    from sglang_amd.quantization.fp8_kernel import sglang_per_token_group_quant_fp8

    g = torch.Generator().manual_seed(0)
    w = torch.randn(N, K, generator=g).to(FP8).to(dev)
    ws = (torch.rand(N // 128, K // 128, generator=g) + 0.1).to(dev)
    packed = torch.full((N, 4), 120, dtype=torch.uint8).view(torch.int32).to(dev)
    rows = torch.ones(N, 1, device=dev)
    block = [128, 128]

    def quantised(x, bias):
        q, s = sglang_per_token_group_quant_fp8(x, 128)
        return fu.aiter_w8a8_block_fp8_linear(q, w, block, ws, s, bias)

    return {
        "cutlass": lambda x, b: fu.cutlass_w8a8_block_fp8_linear_with_fallback(x, w, block, ws, None, b),
        "triton": lambda x, b: fu.triton_w8a8_block_fp8_linear(x, w, block, ws, None, b),
        "deepgemm": lambda x, b: fu.deepgemm_w8a8_block_fp8_linear_with_fallback(x, w, block, packed, None, b),
        "aiter": lambda x, b: fu.aiter_w8a8_block_fp8_linear(x, w, block, ws, None, b),
        "quantised": quantised,
        "rows": lambda x, b: fu.apply_fp8_linear(x, w.t(), rows, bias=b, use_per_token_if_dynamic=True),
    }


def _operands(dev):
    g = torch.Generator().manual_seed(1)
    return torch.randn(M, K, generator=g).bfloat16().to(dev), torch.randn(N, generator=g).bfloat16().to(dev)


def test_vmap_over_the_bias(dev, linears):
    x, bias = _operands(dev)
    out = torch.func.vmap(lambda b: linears["rows"](x, b))(torch.stack([bias, -bias]))
    assert torch.equal(out, torch.stack([linears["rows"](x, bias), linears["rows"](x, -bias)]))


def test_a_subclass_gets_its_own_type_back(dev, linears):
    from sglang_amd.quantization.fp8_kernel import sglang_per_token_group_quant_fp8

    class Tagged(torch.Tensor):
        pass

    x, _ = _operands(dev)
    q, _ = sglang_per_token_group_quant_fp8(x.as_subclass(Tagged), 128)
    assert type(q) is Tagged and type(linears["cutlass"](x.as_subclass(Tagged), None)) is Tagged


LINEARS = ["cutlass", "triton", "deepgemm", "aiter", "quantised", "rows"]


@pytest.mark.parametrize("name", LINEARS)
def test_a_bias_that_requires_grad(dev, linears, name):
    """Adding the bias to the GEMM's output records it: its gradient is the number of rows.  The row-scaled operator adds
    it inside and has no backward: its output says that it needs one."""
    x, bias = _operands(dev)
    plain = linears[name](x, bias)
    assert not plain.requires_grad
    bias.requires_grad_()
    out = linears[name](x, bias)
    assert out.requires_grad and torch.equal(out.detach(), plain)
    if name != "rows":
        out.sum().backward()
        assert torch.equal(bias.grad, torch.full_like(bias, M))
    with torch.no_grad():
        assert not linears[name](x, bias).requires_grad


@pytest.mark.parametrize("name", LINEARS[:-1])
def test_forward_mode_over_the_bias(dev, linears, name):
    import torch.autograd.forward_ad as forward_ad

    x, bias = _operands(dev)
    tangent = torch.arange(N, device=dev).bfloat16()
    with forward_ad.dual_level():
        out = linears[name](x, forward_ad.make_dual(bias, tangent))
        assert torch.equal(forward_ad.unpack_dual(out).tangent, tangent.expand(M, N))


def _moe(dev):
    """(hidden, tensors by name, f(hidden, tensors, **runner options)) of a small block-scaled layer."""
    from sglang_amd.moe_runner import MoeRunnerConfig, fused_moe

    g = torch.Generator().manual_seed(2)
    experts, hidden, inner, topk = 4, 256, 128, 2
    t = dict(w1=torch.randn(experts, 2 * inner, hidden, generator=g).to(FP8),
             w2=torch.randn(experts, hidden, inner, generator=g).to(FP8),
             w1_scale=torch.rand(experts, 2, 2, generator=g) + 0.1, w2_scale=torch.rand(experts, 2, 1, generator=g) + 0.1,
             topk_weights=torch.rand(M, topk, generator=g))
    t = {name: v.to(dev) for name, v in t.items()}
    ids = torch.stack([torch.randperm(experts, generator=g)[:topk] for _ in range(M)]).int().to(dev)

    def layer(h, t, **runner):
        return fused_moe(h, t["w1"], t["w2"], (t["topk_weights"], ids, None), MoeRunnerConfig(**runner), use_fp8_w8a8=True,
                         w1_scale=t["w1_scale"], w2_scale=t["w2_scale"], block_shape=[128, 128])

    return torch.randn(M, hidden, generator=g).bfloat16().to(dev), t, layer


@pytest.mark.parametrize("activation", ["silu", "gelu"])  # the layer as one native call, and step by step
@pytest.mark.parametrize("name", ["topk_weights", "w1", "w2_scale", "hidden"])
def test_moe_layer_says_that_it_has_no_backward(dev, name, activation):
    h, t, layer = _moe(dev)
    plain = layer(h, t, inplace=False, activation=activation)
    assert not plain.requires_grad
    (h if name == "hidden" else t[name]).requires_grad_()
    out = layer(h, t, inplace=False, activation=activation)
    assert torch.equal(out.detach(), plain)
    with pytest.raises(RuntimeError, match="no autograd formula"):
        out.sum().backward()
    with torch.no_grad():
        assert not layer(h, t, inplace=False, activation=activation).requires_grad


@pytest.mark.parametrize("activation", ["silu", "gelu"])
def test_moe_layer_in_place_counts_as_a_write(dev, activation):
    """A product that saved the hidden states for its backward must not use them after the layer overwrote them."""
    h, t, layer = _moe(dev)
    plain = layer(h, t, inplace=False, activation=activation)
    before = h._version
    scale = torch.ones(256, dtype=h.dtype, device=dev, requires_grad=True)
    product = h * scale
    assert h._version == before
    assert layer(h, t, inplace=True, activation=activation) is h and torch.equal(h, plain)
    assert h._version > before
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        product.sum().backward()


@pytest.mark.parametrize("activation", ["silu", "gelu"])
def test_moe_layer_in_place_on_inference_tensors(dev, activation):
    h, t, layer = _moe(dev)
    plain = layer(h, t, inplace=False, activation=activation)
    with torch.inference_mode():
        inner = h.clone()
        assert torch.equal(layer(inner, t, inplace=True, activation=activation), plain)
        other = h.clone()
    assert torch.equal(layer(other, t, inplace=True, activation=activation), plain)  # outside the mode
