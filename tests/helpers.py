"""Shared test plumbing: numpy views of a synthetic case, error metrics."""
import numpy as np
import torch


def to_np_f32(t):
    return t.detach().float().cpu().numpy()


def case_np(case):
    """Numpy view of a case from ipex_amd.utils.synthetic for the oracle."""
    return dict(
        x=to_np_f32(case["x"]),
        qw=(case["qweight"].view(torch.uint8) if case["qweight"].dtype == torch.float8_e4m3fn else case["qweight"])
        .cpu()
        .numpy(),
        scales=to_np_f32(case["scales"]),
        zps=None if case["zeros"] is None else to_np_f32(case["zeros"]),
        bias=None if case["bias"] is None else to_np_f32(case["bias"]),
    )


def rel_l2(a, b):
    a = np.asarray(a, dtype=np.float64)
    b = np.asarray(b, dtype=np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


def max_abs(a, b):
    return float(np.max(np.abs(np.asarray(a, dtype=np.float64) - np.asarray(b, dtype=np.float64))))


def bf16_ulp_diff(a, b):
    """|difference| in bf16 ulps between two float32 arrays holding bf16 values."""
    ia = (np.asarray(a, dtype=np.float32).view(np.uint32) >> 16).astype(np.int64)
    ib = (np.asarray(b, dtype=np.float32).view(np.uint32) >> 16).astype(np.int64)
    # map sign-magnitude to a monotone integer line
    ia = np.where(ia & 0x8000, 0x8000 - ia, ia)
    ib = np.where(ib & 0x8000, 0x8000 - ib, ib)
    return np.abs(ia - ib)


def make_context(case, lowp_mode, act_quant_mode=-1, device="cuda", cache=False):
    from ipex_amd import ops

    return ops.WoqLinearOpContext(
        case["qweight"].to(device),
        case["weight_dtype"],
        [case["N"], case["K"]],
        case["scales"].to(device),
        None if case["zeros"] is None else case["zeros"].to(device),
        None if case["bias"] is None else case["bias"].to(device),
        None,
        None,
        case["group_size"],
        lowp_mode,
        act_quant_mode,
        cache,
    )


def make_torch_context(case, lowp_mode, act_quant_mode=-1, device="cuda", cache=False, g_idx=None):
    """The registered custom class (torch.classes.ipex_prepack.WoqLinearOpContext) for a synthetic case,
    made by the registered prepack operator."""
    import torch
    import ipex_amd  # noqa: F401

    return torch.ops.ipex_prepack.weight_only_qlinear_prepack(
        case["qweight"].to(device),
        case["weight_dtype"],
        [case["N"], case["K"]],
        case["scales"].to(device),
        None if case["zeros"] is None else case["zeros"].to(device),
        None if case["bias"] is None else case["bias"].to(device),
        g_idx,
        None,
        case["group_size"],
        lowp_mode,
        act_quant_mode,
        cache,
    )


def scratch_written(ctx, x):
    """Whether woq_hip_linear, called with the scratch that the library asks for, writes any of it: the quantized activations of
    lowp_mode INT8, the partial tiles of workgroups that share K.  ``ctx``: a context of make_context."""
    import ctypes

    from ipex_amd import _kernels, _lib

    lib = _lib.load()
    (N, K), M = ctx.weight_shape_, x.shape[0]
    ptr = lambda t: None if t is None else t.data_ptr()
    need = lib.woq_hip_linear_workspace_bytes(M, K, ctx.lowp_mode_, ctx.act_quant_mode_, ctx.group_size_)
    need = (need + 255) // 256 * 256 + lib.woq_hip_linear_auto_split_k_workspace_bytes(M, K, N, ctx.lowp_mode_)
    scratch = torch.full((max(need, 1),), 0xA5, dtype=torch.uint8, device=x.device)
    counters = torch.zeros(512, dtype=torch.int32, device=x.device)
    out = torch.empty(M, N, dtype=x.dtype, device=x.device)
    p = _lib.LinearParams()
    p.struct_size = ctypes.sizeof(_lib.LinearParams)
    p.x, p.x_dtype, p.out, p.out_dtype = ptr(x), _kernels._ACT_CODE[x.dtype], ptr(out), _kernels._ACT_CODE[x.dtype]
    p.M, p.K, p.N = M, K, N
    p.qweight, p.weight_dtype, p.group_size = ptr(ctx.at_weight_), ctx.weight_dtype_, ctx.group_size_
    p.scales_f32, p.scales_f16, p.scales_bf16 = (ptr(t) for t in ctx.scales_list_)
    p.zeros_u8, p.bias = ptr(ctx.zeros_u8_), ptr(ctx.bias_f32_)
    p.scale_zero_f16x2, p.scale_zero_bf16 = ptr(ctx.scale_zero_f16x2_), ptr(ctx.scale_zero_bf16_)
    p.lowp_mode, p.act_quant_mode = ctx.lowp_mode_, ctx.act_quant_mode_
    p.workspace, p.workspace_bytes, p.split_k_counters = (ptr(scratch), need, ptr(counters)) if need else (None, 0, None)
    p.stream = torch.cuda.current_stream().cuda_stream
    _lib.check(lib.woq_hip_linear(ctypes.byref(p)), "woq_linear")
    torch.cuda.synchronize()
    return bool((scratch != 0xA5).any())
