"""PyTorch operator surface of the gfx950 W4A16 library.

Defines (when nothing else has) and implements, for the CUDA dispatch key (= HIP tensors on
PyTorch-ROCm), the operators the reference reaches through `vllm/_custom_ops.py`:

  _C::gptq_marlin_repack, _C::awq_marlin_repack, _C::gptq_marlin_gemm, _C::permute_cols,
  _C::silu_and_mul, _moe_C::moe_wna16_marlin_gemm, _moe_C::moe_align_block_size, _moe_C::moe_sum,
  _moe_C::topk_softmax, _moe_C::batched_moe_align_block_size

with the reference's schemas (csrc/torch_bindings.cpp:118, 312-336; csrc/moe/torch_bindings.cpp:13-23, 63-75),
plus fake (meta) implementations for tracing (reference vllm/_custom_ops.py:553-576, 1179-1218,
2089-2120).  The implementations themselves are native (csrc/torch_ops.cpp), one C-ABI call each.  On ROCm builds of the reference these operator definitions are compiled out
(csrc/torch_bindings.cpp:240, csrc/moe/torch_bindings.cpp:52), which is why they are defined here.

The Python wrappers below keep the names and argument order of the reference's wrappers
(vllm/_custom_ops.py:1167-1303, 2004-2060).  Every implementation calls the HIP library through
its C ABI; there is no fallback.
"""
from collections.abc import Callable

import torch

from . import _lib
from .scalar_type import ScalarType

_lib.load()  # fail loudly at import if the HIP library is missing; the native operators bind to it
from . import _torch_ops as _native  # noqa: E402

_GEMM_SCHEMA = (
    "gptq_marlin_gemm(Tensor a, Tensor? c_or_none, Tensor b_q_weight, Tensor? b_bias_or_none, "
    "Tensor b_scales, Tensor? global_scale, Tensor? b_zeros_or_none, Tensor? g_idx_or_none, "
    "Tensor? perm_or_none, Tensor workspace, int b_q_type, SymInt size_m, SymInt size_n, "
    "SymInt size_k, bool is_k_full, bool use_atomic_add, bool use_fp32_reduce, "
    "bool is_zp_float) -> Tensor")
_MOE_GEMM_SCHEMA = (
    "moe_wna16_marlin_gemm(Tensor! a, Tensor? c_or_none, Tensor! b_q_weight, Tensor? b_bias_or_none, "
    "Tensor! b_scales, Tensor? global_scale, Tensor? b_zeros_or_none, Tensor? g_idx_or_none, "
    "Tensor? perm_or_none, Tensor! workspace, Tensor sorted_token_ids, Tensor! expert_ids, "
    "Tensor! num_tokens_past_padded, Tensor! topk_weights, int moe_block_size, int top_k, "
    "bool mul_topk_weights, bool is_ep, int b_q_type_id, int size_m, int size_n, int size_k, "
    "bool is_full_k, bool use_atomic_add, bool use_fp32_reduce, bool is_zp_float) -> Tensor")

_C_SCHEMAS = {
    "gptq_marlin_gemm": _GEMM_SCHEMA,
    "gptq_marlin_repack": "gptq_marlin_repack(Tensor b_q_weight, Tensor perm, SymInt size_k, SymInt size_n, "
                          "int num_bits) -> Tensor",
    "awq_marlin_repack": "awq_marlin_repack(Tensor b_q_weight, SymInt size_k, SymInt size_n, int num_bits) -> Tensor",
    "permute_cols": "permute_cols(Tensor A, Tensor perm) -> Tensor",
    "silu_and_mul": "silu_and_mul(Tensor! result, Tensor input) -> ()",
}
_MOE_SCHEMAS = {
    "moe_wna16_marlin_gemm": _MOE_GEMM_SCHEMA,
    "moe_align_block_size": "moe_align_block_size(Tensor topk_ids, int num_experts, int block_size, "
                            "Tensor! sorted_token_ids, Tensor! experts_ids, Tensor! num_tokens_post_pad) -> ()",
    "batched_moe_align_block_size": "batched_moe_align_block_size(int max_tokens_per_batch, int block_size, "
                                    "Tensor expert_num_tokens, Tensor! sorted_token_ids, Tensor! experts_ids, "
                                    "Tensor! num_tokens_post_pad) -> ()",
    "moe_sum": "moe_sum(Tensor input, Tensor! output) -> ()",
    "topk_softmax": "topk_softmax(Tensor! topk_weights, Tensor! topk_indices, Tensor! token_expert_indices, "
                    "Tensor gating_output, bool renormalize) -> ()",
}


# ------------------------------------------------------------------------------------- fakes
def _gemm_fake(a, c_or_none, b_q_weight, b_bias_or_none, b_scales, global_scale, b_zeros_or_none,
               g_idx_or_none, perm_or_none, workspace, b_q_type, size_m, size_n, size_k,
               is_k_full=True, use_atomic_add=False, use_fp32_reduce=False, is_zp_float=False):
    return torch.empty((size_m, size_n), device=a.device, dtype=a.dtype)


def _repack_fake(b_q_weight, perm, size_k, size_n, num_bits):
    return torch.empty((size_k // 16, size_n * 16 // (32 // num_bits)), dtype=b_q_weight.dtype, device=b_q_weight.device)


def _awq_repack_fake(b_q_weight, size_k, size_n, num_bits):
    return torch.empty((size_k // 16, size_n * 16 // (32 // num_bits)), dtype=b_q_weight.dtype, device=b_q_weight.device)


def _moe_gemm_fake(a, c_or_none, b_q_weight, b_bias_or_none, b_scales, global_scale, b_zeros_or_none,
                   g_idx_or_none, perm_or_none, workspace, sorted_token_ids, expert_ids, num_tokens_past_padded,
                   topk_weights, moe_block_size, top_k, mul_topk_weights, is_ep, b_q_type_id, size_m, size_n,
                   size_k, is_full_k, use_atomic_add, use_fp32_reduce, is_zp_float):
    return torch.empty((size_m * top_k, size_n), dtype=a.dtype, device=a.device)


_FAKES = {
    "_C": {
        "gptq_marlin_gemm": _gemm_fake,
        "gptq_marlin_repack": _repack_fake,
        "awq_marlin_repack": _awq_repack_fake,
        "permute_cols": lambda A, perm: torch.empty_like(A, memory_format=torch.contiguous_format),
        "silu_and_mul": lambda result, input: None,
    },
    "_moe_C": {
        "moe_wna16_marlin_gemm": _moe_gemm_fake,
        "moe_align_block_size": lambda *a: None,
        "batched_moe_align_block_size": lambda *a: None,
        "moe_sum": lambda input, output: None,
        "topk_softmax": lambda *a: None,
    },
}
# Operators of this library's own: the MoE GEMM with a fused epilogue (no counterpart in the reference, which runs
# silu_and_mul and moe_sum as separate launches).  c, workspace and zero_fill are written.
_OWN_SCHEMAS = {
    "moe_marlin_gemm_fused": (
        "moe_marlin_gemm_fused(Tensor a, Tensor(a!) c, Tensor b_q_weight, Tensor? b_bias_or_none, Tensor b_scales, "
        "Tensor? global_scale, Tensor? b_zeros_or_none, Tensor? g_idx_or_none, Tensor? perm_or_none, "
        "Tensor(b!) workspace, Tensor sorted_token_ids, Tensor expert_ids, Tensor num_tokens_past_padded, "
        "Tensor topk_weights, int moe_block_size, int top_k, bool mul_topk_weights, int b_q_type_id, int size_m, "
        "int size_n, int size_k, bool is_full_k, bool silu_and_mul, int sum_top_k, Tensor(c!)? zero_fill) -> ()"),
}
_FAKES["w4a16"] = {"moe_marlin_gemm_fused": lambda *a: None}
_SCHEMAS = {"_C": _C_SCHEMAS, "_moe_C": _MOE_SCHEMAS, "w4a16": _OWN_SCHEMAS}
_libs: list = []          # keep torch.library.Library objects alive
REGISTERED: list[str] = []  # "ns::op" names this module defined and implemented


def _has_op(ns: str, name: str) -> bool:
    try:
        return hasattr(getattr(torch.ops, ns), name)
    except (AttributeError, RuntimeError):
        return False


def _register() -> None:
    for ns, ops_ in _FAKES.items():
        frag = torch.library.Library(ns, "FRAGMENT")
        _libs.append(frag)
        for name, fake in ops_.items():
            if _has_op(ns, name):
                continue  # somebody else (a CUDA build of the reference) already provides it
            frag.define(_SCHEMAS[ns][name], tags=(torch.Tag.needs_fixed_stride_order,))
            _native.register_impl(ns, name)
            torch.library.register_fake(f"{ns}::{name}", fake, lib=frag)
            REGISTERED.append(f"{ns}::{name}")


_register()

# (x, qweight, scales, zeros, g_idx, sort_indices, workspace, type id, N, K, is_k_full, bias, use_fp32_reduce) -> output, or
# None when the call has to go through the dispatcher
eager_linear = _native.linear if "_C::gptq_marlin_gemm" in REGISTERED else lambda *args: None
# the same for routing, (gating_output, topk, renormalize) -> (weights, ids, source rows), and for a whole MoE layer (arguments at
# py_moe in torch_ops.cpp)
eager_topk = _native.topk if "_moe_C::topk_softmax" in REGISTERED else lambda *args: None
eager_moe = (_native.moe if {"_moe_C::moe_align_block_size", "_moe_C::moe_wna16_marlin_gemm", "_moe_C::moe_sum"} <= set(REGISTERED)
             else lambda *args: None)


# ----------------------------------------------------------------- wrappers (reference names)
def gptq_marlin_repack(b_q_weight: torch.Tensor, perm: torch.Tensor, size_k: int, size_n: int,
                       num_bits: int) -> torch.Tensor:
    return torch.ops._C.gptq_marlin_repack(b_q_weight, perm, size_k, size_n, num_bits)


def awq_marlin_repack(b_q_weight: torch.Tensor, size_k: int, size_n: int, num_bits: int) -> torch.Tensor:
    return torch.ops._C.awq_marlin_repack(b_q_weight, size_k, size_n, num_bits)


_STACK_ROWS = 1 << 23  # rows one launch of a repack kernel takes for a stack of experts (its grid allows twice that)


def _repack_stack(repack: Callable, b_q_weight: torch.Tensor, size_k: int, size_n: int, num_bits: int) -> torch.Tensor:
    """[E, rows, cols] checkpoint weights -> [E, K/16, N * bits / 2].  A k-tile never crosses an expert, so a stack of
    experts is one weight of E * K rows to the repack kernels: one launch instead of a launch and a copy per expert
    (128 experts of 2048 x 1536 and 768 x 2048: 4.85 ms, bound by the launches, against 0.13 ms, 4.6 TB/s)."""
    num_experts = b_q_weight.shape[0]
    assert size_k % 16 == 0
    step = max(1, _STACK_ROWS // max(size_k, 1))
    parts = []
    for e in range(0, num_experts, step):
        w = b_q_weight[e:e + step]
        parts.append(repack(w.reshape(-1, w.shape[2]), e, w.shape[0]))
    shape = (num_experts, size_k // 16, size_n * (num_bits // 2))
    if not parts:
        return torch.empty(shape, device=b_q_weight.device, dtype=b_q_weight.dtype)
    return (parts[0] if len(parts) == 1 else torch.cat(parts)).view(shape)


def gptq_marlin_moe_repack(b_q_weight: torch.Tensor, perm: torch.Tensor, size_k: int, size_n: int,
                           num_bits: int) -> torch.Tensor:
    """Repack of every expert, as vllm/_custom_ops.py:1221-1239."""
    def repack(w, e, count):
        order = perm[e:e + count]
        if order.numel():  # row numbers inside the stack
            order = order + size_k * torch.arange(count, dtype=order.dtype, device=order.device).unsqueeze(1)
        return torch.ops._C.gptq_marlin_repack(w, order.reshape(-1), count * size_k, size_n, num_bits)
    return _repack_stack(repack, b_q_weight, size_k, size_n, num_bits)


def awq_marlin_moe_repack(b_q_weight: torch.Tensor, perm: torch.Tensor, size_k: int, size_n: int,
                          num_bits: int) -> torch.Tensor:
    """Repack of every expert, as vllm/_custom_ops.py:1242-1260 (`perm` is unused there too)."""
    return _repack_stack(lambda w, e, count: torch.ops._C.awq_marlin_repack(w, count * size_k, size_n, num_bits),
                         b_q_weight, size_k, size_n, num_bits)


def gptq_marlin_gemm(a, c, b_q_weight, b_bias, b_scales, global_scale, b_zeros, g_idx, perm, workspace,
                     b_q_type: ScalarType, size_m: int, size_n: int, size_k: int, is_k_full: bool = True,
                     use_atomic_add: bool = False, use_fp32_reduce: bool = False,
                     is_zp_float: bool = False) -> torch.Tensor:
    return torch.ops._C.gptq_marlin_gemm(a, c, b_q_weight, b_bias, b_scales, global_scale, b_zeros, g_idx, perm,
                                         workspace, b_q_type.id, size_m, size_n, size_k, is_k_full,
                                         use_atomic_add, use_fp32_reduce, is_zp_float)


def moe_wna16_marlin_gemm(input, output, b_qweight, b_bias, b_scales, global_scale, b_qzeros, g_idx, perm,
                          workspace, sorted_token_ids, expert_ids, num_tokens_past_padded, topk_weights,
                          moe_block_size: int, top_k: int, mul_topk_weights: bool, is_ep: bool,
                          b_q_type: ScalarType, size_m: int, size_n: int, size_k: int, is_k_full: bool,
                          use_atomic_add: bool, use_fp32_reduce: bool, is_zp_float: bool) -> torch.Tensor:
    return torch.ops._moe_C.moe_wna16_marlin_gemm(
        input, output, b_qweight, b_bias, b_scales, global_scale, b_qzeros, g_idx, perm, workspace,
        sorted_token_ids, expert_ids, num_tokens_past_padded, topk_weights, moe_block_size, top_k,
        mul_topk_weights, is_ep, b_q_type.id, size_m, size_n, size_k, is_k_full, use_atomic_add,
        use_fp32_reduce, is_zp_float)


def moe_marlin_gemm_fused(a, c, b_qweight, b_bias, b_scales, global_scale, b_qzeros, g_idx, perm, workspace,
                          sorted_token_ids, expert_ids, num_tokens_past_padded, topk_weights, moe_block_size: int,
                          top_k: int, mul_topk_weights: bool, b_q_type: ScalarType, size_m: int, size_n: int,
                          size_k: int, is_k_full: bool, silu_and_mul: bool = False, sum_top_k: int = 0,
                          zero_fill: torch.Tensor | None = None) -> None:
    """The MoE GEMM writing through a fused epilogue into `c`: silu_and_mul -> c [size_m * top_k, size_n / 2];
    sum_top_k = 2 -> c [size_m * top_k / 2, size_n] (zero on entry) receives each token's two rows added up;
    zero_fill: a tensor this launch also clears."""
    torch.ops.w4a16.moe_marlin_gemm_fused(
        a, c, b_qweight, b_bias, b_scales, global_scale, b_qzeros, g_idx, perm, workspace, sorted_token_ids,
        expert_ids, num_tokens_past_padded, topk_weights, moe_block_size, top_k, mul_topk_weights, b_q_type.id,
        size_m, size_n, size_k, is_k_full, silu_and_mul, sum_top_k, zero_fill)


def batched_moe_align_block_size(max_tokens_per_batch: int, block_size: int, expert_num_tokens: torch.Tensor,
                                 sorted_ids: torch.Tensor, expert_ids: torch.Tensor,
                                 num_tokens_post_pad: torch.Tensor) -> None:
    torch.ops._moe_C.batched_moe_align_block_size(max_tokens_per_batch, block_size, expert_num_tokens, sorted_ids,
                                                  expert_ids, num_tokens_post_pad)


def permute_cols(a: torch.Tensor, perm: torch.Tensor) -> torch.Tensor:
    return torch.ops._C.permute_cols(a, perm)


def silu_and_mul(out: torch.Tensor, x: torch.Tensor) -> None:
    torch.ops._C.silu_and_mul(out, x)


def moe_align_block_size(topk_ids, num_experts, block_size, sorted_token_ids, experts_ids,
                         num_tokens_post_pad) -> None:
    torch.ops._moe_C.moe_align_block_size(topk_ids, num_experts, block_size, sorted_token_ids, experts_ids,
                                          num_tokens_post_pad)


def moe_sum(input: torch.Tensor, output: torch.Tensor) -> None:
    torch.ops._moe_C.moe_sum(input, output)


def topk_softmax(topk_weights: torch.Tensor, topk_ids: torch.Tensor, token_expert_indices: torch.Tensor,
                 gating_output: torch.Tensor, renormalize: bool = False) -> None:
    torch.ops._moe_C.topk_softmax(topk_weights, topk_ids, token_expert_indices, gating_output, renormalize)
