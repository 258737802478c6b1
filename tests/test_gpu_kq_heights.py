"""Tall K-split tiles (gemm_kq.hip) of 80, 96, 112 and 128 rows x 256 columns: whole problems unsplit and with K in two or three equal or
unequal splits across workgroups, and the trailing strips of a prefill launch.  And tiles of 32, 48 and 64 rows x 128 columns whose K parts
are single wavefronts.

Operands are the 16-bit rounded weights (with one scale per column: the integers, the scale applied to the fp32 sum), so results are held
to the float64 product with those.  What is left is the rounding of the result: 2^-11 / sqrt(12) of a value at the bottom of a binade of
fp16, half of that at the top, 2.08e-4 of the root mean square on bell-shaped results (bf16: eight times that); fp32 sums over K <= 5888
add less than 2e-5.  Bounds: 2.3e-4 and 1.75e-3."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [
    # (M, K, N)
    (333, 512, 12352),    # 80 rows, last strip one n-tile of 64 columns
    (212, 2304, 9728),    # ... K in 40 + 32 k-steps
    (556, 768, 9536),     # 96 rows
    (161, 2816, 12352),   # ... K in 48 + 40 k-steps
    (333, 2048, 16448),   # 112 rows
    (508, 3840, 4224),    # ... three splits of 40
    (356, 3840, 6528),    # 128 rows, three splits of 40
    (932, 1792, 17536),   # prefill kernel on the first strips, 80-row tiles on the rest
    (1260, 1280, 13952),
    (88, 5888, 11456),    # fewer than 128 rows: 96 rows, five splits
]
MODES = [
    # (dtype, format, group, act-order)
    (torch.float16, "uint4b8", 128, False),
    (torch.float16, "uint4", 32, False),
    (torch.bfloat16, "uint4b8", 64, False),
    (torch.float16, "uint4", -1, False),
    (torch.float16, "uint4b8", 128, True),
]

# tiles whose eight K parts are single wavefronts
PRIVATE_SHAPES = [
    (29, 4096, 28672),    # 32 rows
    (37, 4096, 28672),    # 48 rows
    (135, 1024, 10816),   # ... one iteration per part, last tile one n-tile
    (162, 2560, 1344),    # ... K in 28 + 28 + 24 k-steps: parts of 0, 4 and 8
    (149, 4096, 3968),    # ... two splits
    (60, 4096, 28672),    # 64 rows
]
PRIVATE_MODES = [
    (torch.float16, "uint4b8", 128, False),
    (torch.float16, "uint4", 128, False),
    (torch.bfloat16, "uint4b8", 128, False),
    (torch.bfloat16, "uint4", -1, False),
    (torch.float16, "uint4b8", -1, False),
    (torch.float16, "uint4b8", 256, False),
    (torch.float16, "uint4b8", 128, True),
    # scales with every k-step
    (torch.float16, "uint4b8", 64, False),
    (torch.float16, "uint4", 32, False),
    (torch.bfloat16, "uint4b8", 32, False),
    (torch.bfloat16, "uint4", 64, False),
]


@pytest.fixture
def workspace(dev):
    from vllm_amd.marlin_utils import marlin_make_workspace_new
    return marlin_make_workspace_new(dev)


def _layer(k, n, fmt, group, dtype, act_order, dev, seed=0):
    """Marlin operands and the weights the kernels multiply with, in float64."""
    from vllm_amd.marlin_utils import marlin_permute_scales, marlin_zero_points
    from vllm_amd.marlin_utils_test import quantize_weights
    from vllm_amd.quant_utils import gptq_pack
    from vllm_amd.scalar_type import scalar_types as st
    import vllm_amd.ops as ops
    g = torch.Generator(device=dev).manual_seed(seed)
    w = (torch.randn(k, n, generator=g, device=dev) * 0.02).to(dtype)
    wtype, gs = (st.uint4, st.uint4b8)[fmt == "uint4b8"], k if group == -1 else group
    w_ref, q, s, z = quantize_weights(w, wtype, gs, zero_points=fmt == "uint4", rule="absmax")
    ref = w_ref.double()
    if group == -1:
        ref = (q.double() - (8 if z is None else z.double())) * s.double()
    e = torch.empty(0, dtype=torch.int32, device=dev)
    g_idx = perm = e
    if act_order:
        order = torch.randperm(k, generator=g, device=dev)  # row i of the sorted weight is K row order[i]
        by_row = torch.empty_like(order)
        by_row[order] = torch.arange(k, device=dev)
        q, ref = q[by_row], ref[by_row]
        perm = order.int()
        g_idx = torch.div(torch.arange(k, device=dev), gs, rounding_mode="floor").int()
    mq = ops.gptq_marlin_repack(gptq_pack(q, 4, k, n), perm, k, n, 4)
    mz = e if z is None else marlin_zero_points(z, k // gs, n, 4)
    return mq, marlin_permute_scales(s, k, n, gs), mz, g_idx, perm, wtype, ref


def _run(a, layer, n, k, workspace, bias=None):
    import vllm_amd.ops as ops
    mq, ms, mz, g_idx, perm, wtype, _ = layer
    return ops.gptq_marlin_gemm(a, None, mq, bias, ms, None, mz, g_idx, perm, workspace, wtype, a.shape[0], n, k, True, False, True, False)


def _rel(out, ref):
    return float((out.double() - ref).norm() / ref.norm())


@pytest.mark.parametrize("m,k,n,dtype,fmt,group,act_order",
                         [s + t for s in SHAPES for t in MODES] + [s + t for s in PRIVATE_SHAPES for t in PRIVATE_MODES])
def test_against_float64(dev, workspace, m, k, n, dtype, fmt, group, act_order):
    print(f"kq heights m={m} k={k} n={n} {dtype} {fmt} group={group} act_order={act_order}", flush=True)
    from vllm_amd.marlin_utils import marlin_permute_bias
    bound = 2.3e-4 if dtype == torch.float16 else 1.75e-3
    layer = _layer(k, n, fmt, group, dtype, act_order, dev)
    g = torch.Generator(device=dev).manual_seed(m)
    a = torch.randn(m, k + 64, generator=g, device=dev).to(dtype)[:, 32:32 + k]  # a strided view
    ref = a.double() @ layer[-1]
    out = _run(a, layer, n, k, workspace)
    assert _rel(out, ref) < bound
    assert torch.equal(out, _run(a.contiguous(), layer, n, k, workspace))
    bias = torch.randn(n, generator=g, device=dev).to(dtype)
    assert _rel(_run(a, layer, n, k, workspace, marlin_permute_bias(bias)), ref + bias.double()) < bound
    assert int(workspace.abs().sum()) == 0


@pytest.mark.parametrize("m,k,n", [(508, 3840, 4224), (356, 3840, 6528)])
def test_entry_point_without_scratch(dev, m, k, n):
    """A caller of the C entry point without scratch still gets a plan that needs none."""
    from vllm_amd import _lib
    lib = _lib.load()
    layer = _layer(k, n, "uint4b8", 128, torch.float16, False, dev)
    a = torch.randn(m, k, generator=torch.Generator(device=dev).manual_seed(1), device=dev).half()
    c, ws = torch.zeros(m, n, dtype=torch.float16, device=dev), torch.zeros(4096, dtype=torch.int32, device=dev)
    args = _lib.GemmArgs()
    args.struct_size = ctypes.sizeof(_lib.GemmArgs)
    args.dtype, args.wtype, args.flags = _lib.DTYPE_F16, _lib.WTYPE_U4B8, _lib.F_IS_K_FULL | _lib.F_USE_FP32_REDUCE
    args.a, args.lda, args.c = a.data_ptr(), a.stride(0), c.data_ptr()
    args.b_q_weight, args.b_scales = layer[0].data_ptr(), layer[1].data_ptr()
    args.size_m, args.size_n, args.size_k, args.num_groups = m, n, k, k // 128
    args.workspace, args.workspace_len = ws.data_ptr(), ws.numel()
    assert lib.w4a16_gemm_scratch_bytes(ctypes.byref(args)) > 0
    assert lib.w4a16_marlin_gemm(ctypes.byref(args), ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream)) == 0, lib.w4a16_last_error()
    assert _rel(c, a.double() @ layer[-1]) < 2.3e-4
