"""The work that users of this library have it do, as cases that can be prepared, run and priced one by one.

Five paths, through the entry points that a serving stack calls:

  block_linear   a linear layer with 128x128 block-scaled FP8 weights: activations quantised per 1x128 group, then the
                 block GEMM.  "norm" puts the fused residual-add + RMSNorm + quantisation in front of it instead (the
                 layer input of a decoder block), "scales" is "float" or "ue8m0" (packed power-of-two exponents).
  row_linear     a linear layer with per-channel FP8 or INT8 weights and per-token activation scales.
  moe            a mixture-of-experts layer: softmax top-k router, then the fused experts ("block_fp8", "block_int8",
                 "channel_fp8", "channel_int8").
  moe_grouped    the same layer through the expert-major (permuted rows, grouped GEMM) interface.
  quant          activation quantisation alone, in the layouts that its callers ask for, with or without SiLU*mul.

Decode is few tokens (1 to some tens), prefill hundreds to thousands; sizes are those of the DeepSeek-V3 and
Llama-3-70B layers of the benchmark, and generic ones."""
import math

import torch

from sglang_amd.gemm import int8_scaled_mm
from sglang_amd.moe import topk_softmax
from sglang_amd.moe_runner.base import MoeRunnerConfig
from sglang_amd.moe_runner.cutlass_moe import cutlass_fused_experts_fp8
from sglang_amd.moe_runner.fused_moe import fused_experts
from sglang_amd.quantization.fp8_kernel import sglang_per_token_group_quant_fp8, sglang_per_token_quant_fp8
from sglang_amd.quantization.fp8_utils import (
    aiter_w8a8_block_fp8_linear,
    apply_fp8_linear,
    dispatch_w8a8_block_fp8_linear,
)
from sglang_amd.quantization.fused_fp8_quant import fused_rms_fp8_group_quant
from sglang_amd.quantization.int8_kernel import per_token_quant_int8

BLOCK = [128, 128]
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}

# (n, k) of the benchmark's weights: DeepSeek-V3 gate_up, down, q_b, o_proj; Llama-3-70B qkv, o, gate_up, down
DSV3 = [(36864, 7168), (7168, 18432), (24576, 1536), (7168, 16384)]
LLAMA70B = [(10240, 8192), (8192, 8192), (57344, 8192), (8192, 28672)]


def listed():
    return [
        # one token through an attention output projection: decode of a single request
        dict(name="block_linear_decode_1", path="block_linear", m=1, n=7168, k=16384, dtype="bf16", scales="float", norm=False, bias=False),
        # a small odd decode batch, residual add and RMSNorm in front of the projection
        dict(name="block_linear_norm_decode_23", path="block_linear", m=23, n=24576, k=1536, dtype="bf16", scales="float", norm=True, bias=False),
        # a short prompt (or a large decode batch) of a ragged length, power-of-two scales
        dict(name="block_linear_ue8m0_300", path="block_linear", m=300, n=7168, k=18432, dtype="bf16", scales="ue8m0", norm=False, bias=False),
        # a full prefill chunk through the widest dense weight
        dict(name="block_linear_prefill_4096", path="block_linear", m=4096, n=36864, k=7168, dtype="bf16", scales="float", norm=False, bias=False),
        # per-channel FP8 decode of a few requests
        dict(name="fp8_linear_decode_7", path="row_linear", m=7, n=10240, k=8192, dtype="f16", quant="fp8", bias=False),
        # per-channel INT8 prefill with a bias, ragged length
        dict(name="int8_linear_prefill_1000", path="row_linear", m=1000, n=8192, k=28672, dtype="bf16", quant="int8", bias=True),
        # the MoE layer: one token, an odd decode batch, a full prefill chunk
        dict(name="moe_decode_1", path="moe", tokens=1, experts=256, topk=8, hidden=7168, inter=2048, dtype="bf16", quant="block_fp8"),
        dict(name="moe_decode_37", path="moe", tokens=37, experts=256, topk=8, hidden=7168, inter=2048, dtype="bf16", quant="block_fp8"),
        dict(name="moe_prefill_4096", path="moe", tokens=4096, experts=256, topk=8, hidden=7168, inter=2048, dtype="bf16", quant="block_fp8"),
        # a layer of medium size with per-channel INT8 experts
        dict(name="moe_channel_int8_250", path="moe", tokens=250, experts=64, topk=6, hidden=4096, inter=1536, dtype="bf16", quant="channel_int8"),
        # the expert-major interface with a medium batch
        dict(name="moe_grouped_512", path="moe_grouped", tokens=512, experts=256, topk=8, hidden=7168, inter=2048, dtype="bf16"),
        # SiLU*mul and quantisation between the two projections of a large prefill, packed exponents
        dict(name="quant_silu_ue8m0_8192", path="quant", rows=8192, hidden=18432, dtype="bf16", layout="ue8m0", silu=True),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _times(rng, low, high, step):
    return max(low, min(high, _log(rng, low, high) // step * step))


def draw(rng):
    path = rng.choice(["block_linear"] * 5 + ["row_linear"] * 3 + ["moe"] * 4 + ["moe_grouped"] + ["quant"] * 2)
    dtype = rng.choice(["bf16", "bf16", "bf16", "f16"])
    if path == "block_linear":
        # half of the weights are the benchmark's, the others free; output widths need not fill the last scale block
        n, k = rng.choice(DSV3) if rng.random() < 0.5 else (_times(rng, 512, 36864, 64), _times(rng, 512, 7168, 128))
        scales = rng.choice(["float", "float", "ue8m0"])
        return dict(path=path, m=_log(rng, 1, 4096), n=n, k=k, dtype=dtype, scales=scales,
                    norm=scales == "float" and dtype == "bf16" and k <= 8192 and rng.random() < 0.4, bias=rng.random() < 0.2)
    if path == "row_linear":
        n, k = rng.choice(LLAMA70B) if rng.random() < 0.5 else (_times(rng, 512, 32768, 8), _times(rng, 512, 8192, 16))
        return dict(path=path, m=_log(rng, 1, 2048), n=n, k=k, dtype=dtype, quant=rng.choice(["fp8", "int8"]), bias=rng.random() < 0.5)
    if path == "moe" or path == "moe_grouped":
        experts = rng.choice([8, 16, 32, 64, 128, 256])
        case = dict(path=path, tokens=_log(rng, 1, 4096), experts=experts, topk=rng.randint(1, 8), hidden=_times(rng, 1024, 7168, 128),
                    inter=_times(rng, 256, 2048, 128), dtype=dtype)
        if path == "moe":
            case["quant"] = rng.choice(["block_fp8"] * 4 + ["block_int8", "channel_fp8", "channel_int8"])
            if rng.random() < 0.3:
                case.update(experts=256, topk=8, hidden=7168, inter=2048)
        return case
    layout = rng.choice(["row", "col", "ue8m0", "token_fp8", "token_int8"])
    return dict(path=path, rows=_log(rng, 1, 16384), hidden=_times(rng, 1024, 18432, 128), dtype=dtype, layout=layout,
                silu=layout in ("row", "col", "ue8m0") and rng.random() < 0.4)


class _Maker:
    """Tensors on the GPU from one seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape, dtype=torch.float32, std=1.0):
        return torch.randn(*shape, generator=self.g, device="cuda", dtype=dtype).mul_(std)

    def uniform(self, *shape, low, high):
        return torch.rand(*shape, generator=self.g, device="cuda").mul_(high - low).add_(low)

    def weight(self, *shape, int8=False):
        """8-bit codes of a normally distributed weight whose blocks' largest values fill the range; made slice by
        slice, so that a layer of experts does not need its 16-bit copy in memory."""
        out = torch.empty(shape, device="cuda", dtype=torch.int8 if int8 else torch.float8_e4m3fn)
        flat = out.view(-1)
        peak = 127.0 if int8 else 448.0
        for at in range(0, flat.numel(), 1 << 28):
            part = flat[at:at + (1 << 28)]
            part.copy_(self.normal(part.numel(), dtype=torch.bfloat16, std=peak / 4).clamp_(-peak, peak))
        return out

    def scales(self, *shape):
        # weights of standard deviation near 0.02: a quarter of the code range times the scale
        return self.uniform(*shape, low=1.2e-4, high=2.4e-4)


def _blocks(v):
    return -(-v // 128)


def _prepare_block_linear(case, make):
    m, n, k, dtype = case["m"], case["n"], case["k"], DTYPES[case["dtype"]]
    state = dict(case=case, x=make.normal(m, k, dtype=dtype), w=make.weight(n, k),
                 bias=make.normal(n, dtype=dtype) if case["bias"] else None)
    if case["scales"] == "ue8m0":
        # exponents 2^-13 and 2^-12, four to a word, the words of a block's row repeated for each weight row in it
        words = -(-_blocks(k) // 4)
        e = torch.randint(114, 116, (_blocks(n), words * 4), generator=make.g, device="cuda", dtype=torch.uint8)
        state["ws"] = e.view(torch.int32).repeat_interleave(128, dim=0)[:n].contiguous()
    else:
        state["ws"] = make.scales(_blocks(n), _blocks(k))
    if case["norm"]:
        state["residual"] = make.normal(m, k, dtype=dtype)
        state["gamma"] = make.uniform(k, low=0.5, high=1.5).to(dtype)
    state["linear"] = dispatch_w8a8_block_fp8_linear()
    return state


def _run_block_linear(s):
    if s["case"]["norm"]:
        (q, q_scale), _, _, residual = fused_rms_fp8_group_quant(s["x"], s["gamma"], 1e-6, res1=s["residual"])
        return aiter_w8a8_block_fp8_linear(q, s["w"], BLOCK, s["ws"], input_scale=q_scale, bias=s["bias"]), residual
    return s["linear"](s["x"], s["w"], BLOCK, s["ws"], bias=s["bias"])


def _prepare_row_linear(case, make):
    m, n, k, dtype = case["m"], case["n"], case["k"], DTYPES[case["dtype"]]
    return dict(case=case, x=make.normal(m, k, dtype=dtype), w=make.weight(n, k, int8=case["quant"] == "int8"),
                ws=make.scales(n, 1), bias=make.normal(n, dtype=dtype) if case["bias"] else None)


def _run_row_linear(s):
    if s["case"]["quant"] == "fp8":
        return apply_fp8_linear(s["x"], s["w"].t(), s["ws"], bias=s["bias"], use_per_token_if_dynamic=True)
    q, q_scale = per_token_quant_int8(s["x"])
    return int8_scaled_mm(q, s["w"].t(), q_scale, s["ws"], out_dtype=s["x"].dtype, bias=s["bias"])


def _prepare_moe(case, make):
    t, e, h, i, dtype = case["tokens"], case["experts"], case["hidden"], case["inter"], DTYPES[case["dtype"]]
    quant = case.get("quant", "block_fp8")
    int8 = quant.endswith("int8")
    state = dict(case=case, x=make.normal(t, h, dtype=dtype), logits=make.normal(t, e),
                 w13=make.weight(e, 2 * i, h, int8=int8), w2=make.weight(e, h, i, int8=int8))
    if quant.startswith("block"):
        state.update(s13=make.scales(e, _blocks(2 * i), _blocks(h)), s2=make.scales(e, _blocks(h), _blocks(i)))
    else:
        state.update(s13=make.scales(e, 2 * i, 1), s2=make.scales(e, h, 1))
    state["options"] = dict(use_int8_w8a8=True) if int8 else dict(use_fp8_w8a8=True)
    if quant.startswith("block"):
        state["options"]["block_shape"] = BLOCK
    else:
        state["options"]["per_channel_quant"] = True
    state["config"] = MoeRunnerConfig(num_experts=e, num_local_experts=e, hidden_size=h, intermediate_size_per_partition=i,
                                      top_k=case["topk"], inplace=False)
    return state


def _route(s):
    t, topk = s["case"]["tokens"], s["case"]["topk"]
    weights = torch.empty(t, topk, device="cuda", dtype=torch.float32)
    ids = torch.empty(t, topk, device="cuda", dtype=torch.int32)
    topk_softmax(weights, ids, s["logits"], renormalize=True)
    return weights, ids


def _run_moe(s):
    weights, ids = _route(s)
    return fused_experts(s["x"], s["w13"], s["w2"], (weights, ids, None), s["config"], w1_scale=s["s13"], w2_scale=s["s2"],
                         **s["options"])


def _prepare_moe_grouped(case, make):
    state = _prepare_moe(case, make)
    e, h, i = case["experts"], case["hidden"], case["inter"]
    i32 = dict(device="cuda", dtype=torch.int32)
    i64 = dict(device="cuda", dtype=torch.int64)
    strides = {w: torch.full((e,), w, **i64) for w in (h, 2 * i, i)}
    # what a model keeps for all its layers: strides, pointer tables, offsets, sizes and scratch
    state["kept"] = (strides[h], strides[2 * i], strides[i], strides[h], torch.empty(1 << 24, device="cuda", dtype=torch.uint8),
                     *(torch.empty(e, **i64) for _ in range(5)), torch.empty(e + 1, **i32), torch.empty(e, 3, **i32),
                     torch.empty(e, 3, **i32))
    return state


def _run_moe_grouped(s):
    weights, ids = _route(s)
    return cutlass_fused_experts_fp8(s["x"], s["w13"].transpose(1, 2), s["w2"].transpose(1, 2), s["s13"].transpose(1, 2),
                                     s["s2"].transpose(1, 2), weights, ids, *s["kept"])


def _prepare_quant(case, make):
    width = case["hidden"] * (2 if case["silu"] else 1)
    return dict(case=case, x=make.normal(case["rows"], width, dtype=DTYPES[case["dtype"]]))


def _run_quant(s):
    layout = s["case"]["layout"]
    if layout == "token_int8":
        return per_token_quant_int8(s["x"])
    if layout == "token_fp8":
        return sglang_per_token_quant_fp8(s["x"])
    return sglang_per_token_group_quant_fp8(s["x"], 128, column_major_scales=layout != "row", scale_tma_aligned=layout == "ue8m0",
                                            scale_ue8m0=layout == "ue8m0", fuse_silu_and_mul=s["case"]["silu"])


_PREPARE = dict(block_linear=_prepare_block_linear, row_linear=_prepare_row_linear, moe=_prepare_moe,
                moe_grouped=_prepare_moe_grouped, quant=_prepare_quant)
_RUN = dict(block_linear=_run_block_linear, row_linear=_run_row_linear, moe=_run_moe, moe_grouped=_run_moe_grouped, quant=_run_quant)


def prepare(case, seed):
    return _PREPARE[case["path"]](case, _Maker(seed))


def run(state):
    return _RUN[state["case"]["path"]](state)


def work(case):
    path = case["path"]
    if path in ("block_linear", "row_linear"):
        m, n, k = case["m"], case["n"], case["k"]
        scales = 4 * _blocks(n) * _blocks(k) if path == "block_linear" else 4 * n
        moved = 2 * m * k + n * k + scales + 2 * m * n + (2 * n if case["bias"] else 0)
        if case.get("norm"):
            moved += 4 * m * k + 2 * k
        return dict(bytes=moved, flops=2.0 * m * n * k)
    if path in ("moe", "moe_grouped"):
        t, e, topk, h, i = case["tokens"], case["experts"], case["topk"], case["hidden"], case["inter"]
        active = e * (1.0 - (1.0 - topk / e) ** t)  # experts that at least one token is expected to pick
        scales = 4 * 3 * _blocks(h) * _blocks(i) if case.get("quant", "block_fp8").startswith("block") else 4 * (2 * i + h)
        return dict(bytes=active * (3 * h * i + scales) + 4 * t * h + 4 * t * e, flops=6.0 * t * topk * h * i)
    rows, hidden = case["rows"], case["hidden"]
    per_row = {"row": hidden // 32, "col": hidden // 32, "ue8m0": -(-hidden // 512) * 4}.get(case["layout"], 4)
    return dict(bytes=rows * (hidden * (4 if case["silu"] else 2) + hidden + per_row), flops=0)


def tolerance(case):
    """Quantised bytes and scales are defined to the bit.  A GEMM's 16-bit results differ by its summation order: a
    last place here and there.  The MoE layer quantises its intermediate rows again, and the value that such a
    last place moves across a rounding boundary changes by up to a sixteenth."""
    if case["path"] == "quant":
        return "exact"
    return {"rel": 4e-3, "max": 4e-2} if case["path"].endswith("linear") else {"rel": 1e-2, "max": 1e-1}
