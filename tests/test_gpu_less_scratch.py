"""Calls whose fastest plan asks for more scratch than the GPU has left run on the plan that needs least, with its results."""
import ctypes

import pytest
import torch

from test_gpu_x8 import _c_args, _layer, _rel, _run
from test_gpu_x8_moe import Moe

pytestmark = pytest.mark.gpu


class Limit:
    """`spare` bytes of GPU memory that the allocator may still take (and no free blocks of 4 MiB in what it holds)."""

    def __init__(self, spare):
        self.spare = spare

    def _set(self, spare):
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + spare) / torch.cuda.get_device_properties(0).total_memory)

    def __enter__(self):
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        self._set(0)
        self.held = []
        try:
            while True:
                self.held.append(torch.empty(4 << 20, dtype=torch.uint8, device="cuda"))
        except torch.OutOfMemoryError:
            pass
        self._set(self.spare)

    def __exit__(self, *exc):
        torch.cuda.set_per_process_memory_fraction(1.0)


def _scratch(args, flags=0):
    from vllm_amd import _lib
    lib = _lib.load()
    args.flags |= flags
    need = lib.w4a16_gemm_scratch_bytes(ctypes.byref(args))
    assert need >= 0, lib.w4a16_last_error()
    return need


@pytest.mark.parametrize("fmt,k,n,m", [("uint4", 512, 131072, 2040), ("uint4b8", 8192, 6144, 4224)])  # prepared weights; 8-bit terms
def test_dense(dev, fmt, k, n, m):
    import vllm_amd.ops as ops
    from vllm_amd import _lib
    from vllm_amd.marlin_utils import marlin_make_workspace_new
    layer = _layer(k, n, fmt, 128, dev, seed=4)
    a = torch.randn(m, k, generator=torch.Generator(device=dev).manual_seed(9), device=dev).bfloat16()
    c, workspace = torch.zeros(m, n, dtype=torch.bfloat16, device=dev), marlin_make_workspace_new(dev)
    args = _c_args(_lib, a, c, layer, n, k, k // 128)
    if fmt == "uint4":
        args.wtype, args.b_zeros = _lib.WTYPE_U4, layer[2].data_ptr()
    assert _scratch(args) > 48 << 20
    assert _scratch(args, _lib.F_LESS_SCRATCH) == 0
    stream = ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream)
    assert _lib.load().w4a16_marlin_gemm(ctypes.byref(args), stream) == 0
    want, full = c.clone(), _run(a, layer, n, k, workspace)
    assert not torch.equal(want, full)
    mq, ms, mz, wtype, _, g_idx, perm = layer
    with Limit(24 << 20):
        ops.gptq_marlin_gemm(a, c.zero_(), mq, None, ms, None, mz, g_idx, perm, workspace, wtype, m, n, k, True, False, True, False)
    assert torch.equal(c, want)
    assert torch.equal(_run(a, layer, n, k, workspace), full)
    assert _rel(c, a.double() @ layer[4]) < 2.5e-3


def test_moe_blocks_of_128(dev):
    import vllm_amd.ops as ops
    from vllm_amd.scalar_type import scalar_types
    moe = Moe(dev, 8192, 192, [9000, 40, 3000], 128)
    a = torch.randn(moe.tokens, moe.k, generator=torch.Generator(device=dev).manual_seed(5), device=dev).bfloat16()
    full = moe.gemm(a)
    s, x, t = moe.routing
    c = torch.full_like(full, 7)
    with Limit(100 << 20):  # (the tail tiles' pieces take 48)
        ops.moe_wna16_marlin_gemm(a, c, moe.w, None, moe.s, None, None, moe.g_idx, moe.perm, moe.workspace, s, x, t, moe.weights, moe_block_size=128,
                                  top_k=1, mul_topk_weights=True, is_ep=False, b_q_type=scalar_types.uint4b8, size_m=moe.tokens, size_n=moe.n,
                                  size_k=moe.k, is_k_full=True, use_atomic_add=False, use_fp32_reduce=True, is_zp_float=False)
    ref = moe.reference(a)
    assert not torch.equal(c, full)
    assert float((c.double() - ref).norm() / ref.norm()) < 2.5e-3
