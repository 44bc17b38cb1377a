"""Timed workloads of the weight-only-quantized linear: what a program that serves a language model asks of it.

A case is a dict of plain values.  ``kind`` says what one pass is: ``linear`` (one layer), ``mlp`` (the gated MLP of a
decoder block), ``block`` (every linear of a decoder block) or ``moe`` (a mixture-of-experts layer).  Weights are normal
with a standard deviation of 0.02 and quantized by the package's own helpers (minimum / maximum per group), activations
are N(0, 1), from ``outliers`` on with one entry in a hundred twenty times as large, as large models have them.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath("intel-extension-for-pytorch_amd"))

import ipex_amd  # noqa: E402,F401  (registers the operators)
from ipex_amd.llm.modules import Linear2SiluMul, LinearAdd, LinearGelu, LinearSilu  # noqa: E402
from ipex_amd.llm.modules.linear_fusion import ConcatLinear  # noqa: E402
from ipex_amd.nn.modules import WeightOnlyQuantizedLinear  # noqa: E402
from ipex_amd.quantization import (  # noqa: E402
    WoqActQuantMode,
    WoqLowpMode,
    WoqWeightDtype,
    get_weight_only_quant_qconfig_mapping,
    quantize_per_block,
    quantize_per_channel,
)

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_WEIGHTS = {"int8": WoqWeightDtype.INT8, "int4": WoqWeightDtype.INT4, "nf4": WoqWeightDtype.NF4, "fp8": WoqWeightDtype.FP8}
_LOWP = {"none": WoqLowpMode.NONE, "fp16": WoqLowpMode.FP16, "bf16": WoqLowpMode.BF16, "int8": WoqLowpMode.INT8}


def _linear(name, M, K, N, weight="int4", group=128, lowp="bf16", act_quant="per_batch_sym", act="bf16", sym=False, bias=False,
            act_order=False, cache=False, post="none", outliers=False):
    return dict(name=name, kind="linear", M=M, K=K, N=N, weight=weight, group=group, lowp=lowp, act_quant=act_quant, act=act,
                sym=sym, bias=bias, act_order=act_order, cache=cache, post=post, outliers=outliers)


def listed():
    return [
        # single-stream decode under lowp_mode INT8, the smallest projection of a 4096-wide model: latency and launches
        _linear("decode_m1_lowp_int8", 1, 4096, 4096, lowp="int8"),
        # single-stream decode: the gated MLP of a 4096-wide model (gate, up and down with the residual), INT4 g128
        dict(name="decode_m1_mlp", kind="mlp", M=1, H=4096, I=14336, group=128),
        # sixteen sequences decoded together: all linears of a decoder block with 32 query and 8 key / value heads, INT4 g32
        dict(name="decode_m16_block", kind="block", M=16, H=4096, Q=4096, KV=1024, I=14336, group=32),
        # INT8 with one scale per output channel and a bias: a batch of 32 through the up projection of a 4096 / 11008 MLP
        _linear("decode_m32_int8_bias", 32, 4096, 11008, weight="int8", group=-1, sym=True, bias=True),
        # the default recipe (INT8 per channel, asymmetric, lowp_mode NONE) on an fp32 model, four beams
        _linear("decode_m4_fp32_default", 4, 4096, 11008, weight="int8", group=-1, lowp="none", act="fp32"),
        # prompt of 2048 tokens, INT4 g128
        _linear("prefill_m2048", 2048, 4096, 14336, outliers=True),
        # the same prompt with the activations quantized per token
        _linear("prefill_m2048_lowp_int8", 2048, 4096, 14336, lowp="int8", outliers=True),
        # a chunk of a prompt through a GPTQ checkpoint with activation order, the down projection and its residual
        _linear("chunk_m333_gptq_act_order", 333, 11008, 4096, act_order=True, post="add"),
        # a short prompt through an NF4 model
        _linear("prompt_m77_nf4", 77, 4096, 11008, weight="nf4", group=64, sym=True),
        # a longer prompt through FP8 weights with a scale per 128 input channels
        _linear("prompt_m1000_fp8", 1000, 7168, 4096, weight="fp8", group=128, sym=True),
        # decode of sixteen tokens through 32 experts, top-8
        dict(name="moe_decode_t16", kind="moe", T=16, E=32, topk=8, H=7168, I=2048, group=128),
        # a prompt of 512 tokens through the same layer
        dict(name="moe_prompt_t512", kind="moe", T=512, E=32, topk=8, H=7168, I=2048, group=128),
    ]


_MAX_FLOPS = 2.0 * 2048 * 4096 * 14336


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear"] * 7 + ["mlp", "block", "moe"])
    if kind == "moe":
        H, I, topk = 128 * rng.randint(8, 56), 128 * rng.randint(4, 16), rng.choice([2, 4, 8])
        return dict(kind="moe", T=_log_int(rng, 1, 512), E=rng.choice([8, 16, 32]), topk=topk, H=H, I=I, group=rng.choice([32, 64, 128]))
    if kind == "mlp":
        H, I = 128 * rng.randint(8, 64), 128 * rng.randint(16, 112)
        return dict(kind="mlp", M=min(_log_int(rng, 1, 512), int(_MAX_FLOPS / (6.0 * H * I))), H=H, I=I, group=rng.choice([32, 64, 128]))
    if kind == "block":
        kv = 128 * rng.randint(4, 8)
        H, I = kv * rng.randint(2, 8), 128 * rng.randint(16, 112)
        M = min(_log_int(rng, 1, 512), int(_MAX_FLOPS / (6.0 * H * I + 4.0 * H * (H + kv))))
        return dict(kind="block", M=M, H=H, Q=H, KV=kv, I=I, group=rng.choice([32, 64, 128]))
    weight = rng.choice(["int4"] * 4 + ["int8"] * 2 + ["nf4", "fp8"])
    K = 128 * _log_int(rng, 8, 112)
    N = _log_int(rng, 512, 28672) if rng.random() < 0.4 else 64 * _log_int(rng, 8, 448)
    M = _log_int(rng, 1, 2048)
    act, lowp = "bf16", "bf16"
    group = -1 if weight == "int8" else rng.choice([32, 64, 128, 128])
    if weight == "fp8":
        group = 128
    if weight in ("int4", "int8") and rng.random() < 0.3:
        lowp = "int8"
    elif weight == "int8" and rng.random() < 0.3:
        lowp, act, M = "none", "fp32", min(M, 128)
    elif rng.random() < 0.15:
        lowp, act = "none", "fp16"
    if group < 0 and rng.random() < 0.15:
        K -= 8 * rng.randint(1, 15)  # widths that are no multiple of a tile
    M = max(1, min(M, int(_MAX_FLOPS / (2.0 * K * N))))
    sym = weight in ("nf4", "fp8") or (weight == "int8" and lowp == "int8") or rng.random() < 0.3
    case = _linear("", M, K, N, weight, group, lowp, rng.choice(["per_batch_sym", "per_batch_ic_block_sym"]), act, sym,
                   bias=rng.random() < 0.3, act_order=weight == "int4" and rng.random() < 0.15,
                   cache=lowp == "bf16" and rng.random() < 0.15, post=rng.choice(["none"] * 3 + ["gelu", "silu", "add"]),
                   outliers=rng.random() < 0.3)
    del case["name"]
    return case


class _Source:
    """Random inputs of one state, made on the GPU from its seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, generator=self.g, device="cuda") * std

    def activations(self, M, K, dtype, outliers=False):
        x = self.normal(M, K)
        if outliers:
            x = torch.where(torch.rand(M, K, generator=self.g, device="cuda") < 0.01, x * 20, x)
        return x.to(dtype)

    def quantized(self, N, K, weight, group, sym):
        """(codes, scales, zero points or None) of a normal weight, as a checkpoint holds them."""
        w = self.normal(N, K, std=0.02)
        if weight == "fp8":
            scales = w.view(N, -1, group).abs().amax(-1) / 448
            return (w.view(N, -1, group) / scales.unsqueeze(-1)).view(N, K).to(torch.float8_e4m3fn), scales, None
        if group > 0:
            return quantize_per_block(w, _WEIGHTS[weight], group, sym_quant=sym)
        return quantize_per_channel(w, _WEIGHTS[weight], sym_quant=sym)

    def module(self, K, N, weight="int4", group=128, lowp="bf16", act_quant="per_batch_sym", sym=False, bias=False, act_order=False,
               cache=False):
        qweight, scales, zeros = self.quantized(N, K, weight, group, sym)
        g_idx = None
        if act_order:
            g_idx = (torch.arange(K, device="cuda") // group)[torch.randperm(K, generator=self.g, device="cuda")].to(torch.int32)
        b = self.normal(N, std=0.02) if bias else None
        mod = torch.nn.Linear(K, N, bias=False, device="meta")
        mod.qconfig = get_weight_only_quant_qconfig_mapping(
            weight_dtype=_WEIGHTS[weight], lowp_mode=_LOWP[lowp],
            act_quant_mode=WoqActQuantMode[act_quant.upper()], group_size=group).global_qconfig._replace(cache_weight_for_large_batch=cache)
        return WeightOnlyQuantizedLinear.from_float_and_qweight(mod, qweight, _WEIGHTS[weight], scales, zeros, b, group, g_idx)

    def expert(self, K, N, group):
        qweight, scales, zeros = self.quantized(N, K, "int4", group, False)
        return torch.ops.ipex_prepack.weight_only_qlinear_prepack(
            qweight, int(WoqWeightDtype.INT4), [N, K], scales, zeros, None, None, None, group, int(WoqLowpMode.BF16), -1, False)


def prepare(case, seed):
    src = _Source(seed)
    kind = case["kind"]
    if kind == "linear":
        M, K, N, dtype = case["M"], case["K"], case["N"], _DTYPES[case["act"]]
        mod = src.module(K, N, case["weight"], case["group"], case["lowp"], case["act_quant"], case["sym"], case["bias"], case["act_order"],
                         case["cache"])
        wrap = {"none": lambda m: m, "gelu": LinearGelu, "silu": LinearSilu, "add": LinearAdd}[case["post"]]
        args = [src.activations(M, K, dtype, case["outliers"])]
        if case["post"] == "add":
            args.append(src.activations(M, N, dtype))
        return dict(kind=kind, layer=wrap(mod), args=args)
    if kind == "moe":
        T, E, H, I, group = case["T"], case["E"], case["H"], case["I"], case["group"]
        lists = [[src.expert(H, I, group) for _ in range(E)], [src.expert(H, I, group) for _ in range(E)], [src.expert(I, H, group) for _ in range(E)]]
        logits = src.normal(T, E)
        weights, ids = torch.topk(torch.softmax(logits, -1), case["topk"], -1)
        weights = (weights / weights.sum(-1, keepdim=True)).to(torch.bfloat16)
        return dict(kind=kind, lists=lists, x=src.activations(T, H, torch.bfloat16), ids=ids, weights=weights)
    M, H, I, group = case["M"], case["H"], case["I"], case["group"]
    state = dict(kind=kind, gate_up=Linear2SiluMul(src.module(H, I, group=group), src.module(H, I, group=group)),
                 down=LinearAdd(src.module(I, H, group=group)), x=src.activations(M, H, torch.bfloat16),
                 residual=src.activations(M, H, torch.bfloat16))
    if kind == "block":
        Q, KV = case["Q"], case["KV"]
        state["qkv"] = ConcatLinear([src.module(H, n, group=group) for n in (Q, KV, KV)])
        state["o"] = LinearAdd(src.module(Q, H, group=group))
        state["attention"] = src.activations(M, Q, torch.bfloat16)
    return state


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return state["layer"](*state["args"])
    if kind == "moe":
        return torch.ops.torch_ipex.deepseek_moe_woq(state["x"], state["ids"], *state["lists"], state["weights"], False)
    if kind == "mlp":
        return state["down"](state["gate_up"](state["x"]), state["residual"])
    qkv = state["qkv"](state["x"])
    o = state["o"](state["attention"], state["residual"])  # (attention and the norms are not this package's)
    return [*qkv, o, state["down"](state["gate_up"](state["x"]), o)]


_NF4 = [-1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453, -0.28444138169288635, -0.18477343022823334,
        -0.09105003625154495, 0.0, 0.07958029955625534, 0.16093020141124725, 0.24611230194568634, 0.33791524171829224,
        0.44070982933044434, 0.5626170039176941, 0.7229568362236023, 1.0]


class _Exact(_Source):
    """The same inputs; a layer is the function that its checkpoint stands for, in 64 bits and without the package's kernels."""

    def module(self, K, N, weight="int4", group=128, lowp="bf16", act_quant="per_batch_sym", sym=False, bias=False, act_order=False,
               cache=False):
        q, scales, zeros = self.quantized(N, K, weight, group, sym)
        index = torch.arange(K, device="cuda") // group if group > 0 else torch.zeros(K, dtype=torch.long, device="cuda")
        if act_order:
            index = index[torch.randperm(K, generator=self.g, device="cuda")]
        b = self.normal(N, std=0.02).double() if bias else None
        if weight in ("int4", "nf4"):
            q = torch.stack([q & 15, q >> 4], -1).view(N, -1)[:, :K]
        w = torch.tensor(_NF4, dtype=torch.float64, device="cuda")[q.long()] if weight == "nf4" else q.double()
        if zeros is not None:
            w -= zeros.double().view(N, -1)[:, index]
        elif weight == "int4":
            w -= 8
        w *= scales.double().view(N, -1)[:, index]
        block = min(group, 128) if group > 0 else 128
        while K % block:
            block //= 2
        if lowp != "int8" or block < 32:  # (such widths are not quantized)
            rows = 0
        else:
            rows = K if act_quant == "per_batch_sym" else group if group > 0 else block

        def linear(x):
            if rows:  # what the option asks for: symmetric int8, a scale per row or per (row, block of input channels)
                v = x.view(x.shape[0], -1, rows)
                s = (v.float().abs().amax(-1, keepdim=True) / 127).double()  # (a 32-bit number by the format)
                x = (torch.clamp(torch.round(v / s), -128, 127) * s).view(x.shape)
            y = x @ w.t()
            return y if b is None else y + b

        return linear

    def expert(self, K, N, group):
        return self.module(K, N, group=group)


def exact(case, seed):
    src = _Exact(seed)
    kind, silu = case["kind"], torch.nn.functional.silu
    if kind == "linear":
        M, K, N, dtype = case["M"], case["K"], case["N"], _DTYPES[case["act"]]
        layer = src.module(K, N, case["weight"], case["group"], case["lowp"], case["act_quant"], case["sym"], case["bias"],
                           case["act_order"], case["cache"])
        y = layer(src.activations(M, K, dtype, case["outliers"]).double())
        if case["post"] == "add":
            return y + src.activations(M, N, dtype).double()
        return {"none": lambda v: v, "gelu": torch.nn.functional.gelu, "silu": silu}[case["post"]](y)
    if kind == "moe":
        T, E, H, I, group = case["T"], case["E"], case["H"], case["I"], case["group"]
        gate, up, down = [[src.expert(k, n, group) for _ in range(E)] for k, n in ((H, I), (H, I), (I, H))]
        weights, ids = torch.topk(torch.softmax(src.normal(T, E), -1), case["topk"], -1)
        weights = (weights / weights.sum(-1, keepdim=True)).to(torch.bfloat16).double()
        x = src.activations(T, H, torch.bfloat16).double()
        y = torch.zeros_like(x)
        for e in range(E):
            t, j = torch.where(ids == e)
            y.index_add_(0, t, down[e](silu(gate[e](x[t])) * up[e](x[t])) * weights[t, j].unsqueeze(-1))
        return y
    M, H, I, group = case["M"], case["H"], case["I"], case["group"]
    gate, up, down = src.module(H, I, group=group), src.module(H, I, group=group), src.module(I, H, group=group)
    x, residual = src.activations(M, H, torch.bfloat16).double(), src.activations(M, H, torch.bfloat16).double()
    mlp = down(silu(gate(x)) * up(x))
    if kind == "mlp":
        return mlp + residual
    Q, KV = case["Q"], case["KV"]
    qkv = [src.module(H, n, group=group) for n in (Q, KV, KV)]
    o = src.module(Q, H, group=group)
    attended = o(src.activations(M, Q, torch.bfloat16).double()) + residual
    return [*(f(x) for f in qkv), attended, mlp + attended]


def _weight_bytes(K, N, weight, group, zeros=True):
    code = 0.5 if weight in ("int4", "nf4") else 1.0
    groups = (K + group - 1) // group if group > 0 else 1
    per_group = 2.0 if weight in ("int4", "nf4") else 4.0  # bf16 scales of 4-bit weights, fp32 ones of bytes
    return N * K * code + N * groups * (per_group + (code if zeros else 0.0))


def _active_experts(case):
    """Experts that have tokens, as expected of an even routing."""
    return case["E"] * (1.0 - (1.0 - case["topk"] / case["E"]) ** case["T"])


def work(case):
    kind = case["kind"]
    if kind == "linear":
        M, K, N, size = case["M"], case["K"], case["N"], _DTYPES[case["act"]].itemsize
        nbytes = _weight_bytes(K, N, case["weight"], case["group"], not case["sym"]) + M * (K + N * (2 if case["post"] == "add" else 1)) * size
        return {"bytes": nbytes + (4 * N if case["bias"] else 0), "flops": 2.0 * M * K * N}
    H, I, group = case["H"], case["I"], case["group"]
    mlp_bytes = 2 * _weight_bytes(H, I, "int4", group) + _weight_bytes(I, H, "int4", group)
    if kind == "moe":
        T = case["T"]
        return {"bytes": _active_experts(case) * mlp_bytes + 2.0 * T * H * 2 + T * case["topk"] * 10, "flops": 6.0 * T * case["topk"] * H * I}
    M = case["M"]
    nbytes, flops = mlp_bytes + 3.0 * M * H * 2, 6.0 * M * H * I
    if kind == "block":
        Q, KV = case["Q"], case["KV"]
        nbytes += _weight_bytes(H, Q + 2 * KV, "int4", group) + _weight_bytes(Q, H, "int4", group) + 2.0 * M * (2 * Q + 2 * KV + H)
        flops += 2.0 * M * H * (2 * Q + 2 * KV)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # Measured against exact(), which is the same products in 64 bits over the unrounded weights and scales, a third to a quarter of what
    # is stated: bf16 outputs of one layer 2.5e-3 .. 3.2e-3 (scales, weights and outputs are rounded to bf16), of a chain
    # of layers 4.2e-3 .. 6.3e-3, fp16 outputs 4.3e-4, fp32 1.1e-6.
    if case["kind"] != "linear":
        return {"rel": 1.6e-2}
    return {"rel": {"bf16": 8e-3, "fp16": 2e-3, "fp32": 4e-6}[case["act"]]}
