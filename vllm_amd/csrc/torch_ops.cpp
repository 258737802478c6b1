// PyTorch operators of the library: argument checks (with the reference's messages), output and scratch allocation, one
// call of the C ABI.  Implementations for the CUDA dispatch key (= HIP tensors on PyTorch-ROCm); the schemas and the fake
// implementations are in _custom_ops.py, which also decides which operators this library provides (`register_impl`).
//
// Why native: the 16-row GEMM of a decode projection runs 5.6-10 us, its launch costs the host about 2 us, and the same
// checks written in Python with a ctypes call cost 28 us per call, so every decode call was bound by the host.
//
// `linear`, `topk` and `moe` at the end are direct entries for eager calls on plain GPU tensors; they skip the dispatcher
// (boxing of 18 arguments: 7.1 -> 5.2 us per linear) and return None when anything may want to see the operator (a tensor subclass,
// a function, dispatch or trace mode, the profiler, autograd) or an argument is one the dispatcher would convert: the caller then
// goes through torch.ops.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/grad_mode.h>
#include <ATen/record_function.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/library.h>

#include "../../include/w4a16_gfx950.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

// ScalarType ids (scalar_type.py): exponent:8, mantissa:8, signed:1, bias:32, finite_values_only:1, nan_repr:8
constexpr int64_t type_id(int exponent, int mantissa, int is_signed, int64_t bias, int finite, int64_t nan_repr) {
  return exponent | (mantissa << 8) | (is_signed << 16) | (bias << 17) | ((int64_t)finite << 49) | (nan_repr << 50);
}
constexpr int64_t kUint4 = type_id(0, 4, 0, 0, 0, 1), kUint4b8 = type_id(0, 4, 0, 8, 0, 1),
                  kUint8b128 = type_id(0, 8, 0, 128, 0, 1), kFp8 = type_id(4, 3, 1, 0, 1, 2),
                  kFp4 = type_id(2, 1, 1, 0, 1, 0);

int64_t size_bits(int64_t id) { return (id & 0xff) + ((id >> 8) & 0xff) + ((id >> 16) & 1); }

std::string type_name(int64_t id) {
  const int64_t exponent = id & 0xff, mantissa = (id >> 8) & 0xff, bias = (id >> 17) & 0xffffffff;
  std::string s;
  if (exponent)
    return "float" + std::to_string(size_bits(id)) + "_e" + std::to_string(exponent) + "m" + std::to_string(mantissa);
  s = ((id >> 16) & 1 ? "int" : "uint") + std::to_string(size_bits(id));
  return bias ? s + "b" + std::to_string(bias) : s;
}

int dtype_code(at::ScalarType t) {
  if (t == at::kHalf) return W4A16_DTYPE_F16;
  TORCH_CHECK(t == at::kBFloat16, "gpt_marlin_gemm only supports bfloat16 and float16");
  return W4A16_DTYPE_BF16;
}

int wtype_code(int64_t id, bool has_zp) {
  int code = -1;
  switch (id) {
    case kUint4b8: code = W4A16_WTYPE_U4B8; break;
    case kUint8b128: code = W4A16_WTYPE_U8B128; break;
    case kFp8: code = W4A16_WTYPE_FE4M3; break;
    case kFp4: code = W4A16_WTYPE_FE2M1; break;
    case kUint4:
      TORCH_CHECK(has_zp, "b_q_type must be uint4b8 or uint8b128 when has_zp = False. Got = uint4");
      return W4A16_WTYPE_U4;
    default:
      TORCH_CHECK_NOT_IMPLEMENTED(false, "weight type ", type_name(id),
                                  " is not implemented by the gfx950 W4A16 library (supported: uint4b8, uint8b128, "
                                  "float8_e4m3fn, float4_e2m1f, uint4 with zero points)");
  }
  TORCH_CHECK(!has_zp, "b_q_type must be uint4 or uint8 when has_zp = True. Got = ", type_name(id));
  return code;
}

int64_t pack_factor(int64_t id) {
  const int64_t bits = size_bits(id);
  TORCH_CHECK(bits > 0 && bits <= 32, "bad b_q_type ", id);
  return 32 / bits;
}

void check_rc(int rc) {
  if (rc == W4A16_OK) return;
  TORCH_CHECK_NOT_IMPLEMENTED(rc != W4A16_ENOTIMPL, w4a16_last_error());
  TORCH_CHECK(false, w4a16_last_error());
}

// `Tensor?` arguments arrive as none or as zero-length tensors; both mean absent
const Tensor* present(const OptTensor& t) { return t.has_value() && t->defined() && t->numel() > 0 ? &*t : nullptr; }
const void* data_or_null(const Tensor* t) { return t ? t->const_data_ptr() : nullptr; }
void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

// Every launch runs on its tensors' device; the guard (a pair of runtime calls) is only set up off the current one.
struct OnDevice {
  explicit OnDevice(const Tensor& t) {
    if (c10::hip::current_device() != t.get_device()) guard.reset_device(t.device());
  }
  c10::OptionalDeviceGuard guard;
};

void check_gpu_i32(const Tensor& t, const char* name) {
  TORCH_CHECK(t.is_cuda() && t.is_contiguous() && t.scalar_type() == at::kInt, name, " must be a contiguous int32 GPU tensor");
}

// ------------------------------------------------------------------------------------------------------ repack
Tensor gptq_marlin_repack(const Tensor& b_q_weight, const Tensor& perm, int64_t size_k, int64_t size_n, int64_t num_bits) {
  TORCH_CHECK(num_bits == 4 || num_bits == 8, "num_bits must be 4 or 8. Got = ", num_bits);
  const int64_t pack = 32 / num_bits;
  TORCH_CHECK(size_k % 16 == 0, "size_k = ", size_k, " is not divisible by tile_k_size = 16");
  TORCH_CHECK(size_n % 64 == 0, "size_n = ", size_n, " is not divisible by tile_n_size = 64");
  TORCH_CHECK(b_q_weight.is_cuda() && b_q_weight.is_contiguous(), "b_q_weight is not a contiguous GPU tensor");
  TORCH_CHECK(b_q_weight.scalar_type() == at::kInt, "b_q_weight type is not kInt");
  TORCH_CHECK(b_q_weight.dim() == 2 && b_q_weight.size(0) == size_k / pack && b_q_weight.size(1) == size_n,
              "Shape mismatch: b_q_weight = ", b_q_weight.sizes(), ", size_k = ", size_k, ", size_n = ", size_n);
  TORCH_CHECK(perm.scalar_type() == at::kInt, "perm type is not at::kInt");
  const bool has_perm = perm.numel() != 0;
  if (has_perm)
    TORCH_CHECK(perm.is_cuda() && perm.is_contiguous() && perm.numel() == size_k, "perm must be a contiguous [size_k] GPU tensor");
  Tensor out = at::empty({size_k / 16, size_n * 16 / pack}, b_q_weight.options());
  if (out.numel()) {
    OnDevice on(b_q_weight);
    check_rc(w4a16_gptq_marlin_repack((const uint32_t*)b_q_weight.const_data_ptr(),
                                      has_perm ? (const int32_t*)perm.const_data_ptr() : nullptr,
                                      (uint32_t*)out.mutable_data_ptr(), size_k, size_n, (int)num_bits, stream_of(out)));
  }
  return out;
}

Tensor awq_marlin_repack(const Tensor& b_q_weight, int64_t size_k, int64_t size_n, int64_t num_bits) {
  TORCH_CHECK(num_bits == 4 || num_bits == 8, "num_bits must be 4 or 8. Got = ", num_bits);
  const int64_t pack = 32 / num_bits;
  TORCH_CHECK(size_k % 16 == 0, "size_k = ", size_k, " is not divisible by tile_k_size = 16");
  TORCH_CHECK(size_n % 64 == 0, "size_n = ", size_n, " is not divisible by tile_n_size = 64");
  TORCH_CHECK(b_q_weight.is_cuda() && b_q_weight.is_contiguous(), "b_q_weight is not a contiguous GPU tensor");
  TORCH_CHECK(b_q_weight.scalar_type() == at::kInt, "b_q_weight type is not kInt");
  TORCH_CHECK(b_q_weight.dim() == 2 && b_q_weight.size(0) == size_k && b_q_weight.size(1) == size_n / pack,
              "Shape mismatch: b_q_weight = ", b_q_weight.sizes(), ", size_k = ", size_k, ", size_n = ", size_n);
  Tensor out = at::empty({size_k / 16, size_n * 16 / pack}, b_q_weight.options());
  if (out.numel()) {
    OnDevice on(b_q_weight);
    check_rc(w4a16_awq_marlin_repack((const uint32_t*)b_q_weight.const_data_ptr(), (uint32_t*)out.mutable_data_ptr(), size_k,
                                     size_n, (int)num_bits, stream_of(out)));
  }
  return out;
}

Tensor permute_cols(const Tensor& A, const Tensor& perm) {
  TORCH_CHECK(A.is_cuda() && A.dim() == 2 && A.stride(1) == 1, "A must be a 2-D GPU tensor with unit column stride");
  TORCH_CHECK(A.scalar_type() == at::kHalf || A.scalar_type() == at::kBFloat16, "A must be fp16 or bf16");
  TORCH_CHECK(perm.is_cuda() && perm.scalar_type() == at::kInt && perm.is_contiguous() && perm.numel() == A.size(1),
              "perm must be a contiguous int32 GPU tensor with one entry per column");
  Tensor out = at::empty({A.size(0), A.size(1)}, A.options());
  if (out.numel()) {
    OnDevice on(A);
    check_rc(w4a16_permute_cols(A.const_data_ptr(), (const int32_t*)perm.const_data_ptr(), out.mutable_data_ptr(), A.size(0),
                                A.size(1), A.stride(0), stream_of(A)));
  }
  return out;
}

// -------------------------------------------------------------------------------------------------------- GEMM
// Scratch comes from torch's caching allocator: stream-ordered reuse, given back when `tmp` goes.  Where the GPU has no room for what the fastest
// plan asks for, the call runs on the one that needs least.
void run_gemm(w4a16_gemm_args& args, const Tensor& a) {
  OnDevice on(a);
  auto scratch = [&]() {
    const int64_t need = w4a16_gemm_scratch_bytes(&args);
    if (need < 0) check_rc((int)need);
    return need > 0 ? at::empty({need / 4}, a.options().dtype(at::kFloat)) : Tensor();
  };
  Tensor tmp;
  try {
    tmp = scratch();
  } catch (const c10::OutOfMemoryError&) {
    args.flags |= W4A16_F_LESS_SCRATCH;
    tmp = scratch();
  }
  if (tmp.defined()) args.c_tmp = (float*)tmp.mutable_data_ptr();
  check_rc(w4a16_marlin_gemm(&args, stream_of(a)));
}

// fp4 scales are one byte per (group, column): NVFP4 (group 16) float8_e4m3fn with a global scale, MXFP4 (group 32)
// float8_e8m0fnu; every other type has scales of the activation type and no global scale.
void check_scales(const Tensor& a, const Tensor& b_scales, int64_t q_type, int64_t size_k, int64_t num_groups, const Tensor* gscale,
                  int64_t experts) {
  if (q_type != kFp4) {
    TORCH_CHECK(b_scales.scalar_type() == a.scalar_type(), "scalar type of a and b_scales must match");
    TORCH_CHECK(gscale == nullptr, "global_scale can only be used for nvfp4 format.");
    return;
  }
  const int64_t group = num_groups > 0 && size_k % num_groups == 0 ? size_k / num_groups : 0;
  TORCH_CHECK(group == 16 || group == 32, "float4_e2m1f only supports group_size == 16 (NVFP4) and group_size == 32 (MXFP4)");
  const auto want = group == 16 ? at::kFloat8_e4m3fn : at::kFloat8_e8m0fnu;
  TORCH_CHECK(b_scales.scalar_type() == want, "b_scales must be ", want, " for float4_e2m1f with group_size = ", group);
  if (group == 16) {
    TORCH_CHECK(gscale != nullptr, "the global_scale parameter must be passed for nvfp4 format.");
    TORCH_CHECK(gscale->is_cuda() && gscale->is_contiguous() && gscale->numel() == experts && gscale->scalar_type() == a.scalar_type(),
                "global_scale must hold one element of the activation type", experts > 1 ? " per expert" : "", " on the GPU");
  } else {
    TORCH_CHECK(gscale == nullptr, "global_scale can only be used for nvfp4 format.");
  }
}

void fill_common(w4a16_gemm_args& args, const Tensor& a, const Tensor& c, const Tensor& w, const Tensor* bias, const Tensor& scales,
                 const Tensor* zeros, const Tensor* g_idx, const Tensor* perm, const Tensor* gscale, const Tensor& workspace,
                 int wtype, int64_t m, int64_t n, int64_t k, int64_t groups, int flags) {
  args.struct_size = sizeof(args);
  args.dtype = dtype_code(a.scalar_type());
  args.wtype = wtype;
  args.flags = flags;
  args.a = a.const_data_ptr();
  args.lda = a.stride(0);
  args.c = c.mutable_data_ptr();
  args.b_q_weight = (const uint32_t*)w.const_data_ptr();
  args.b_scales = scales.const_data_ptr();
  args.b_zeros = (const uint32_t*)data_or_null(zeros);
  args.g_idx = (const int32_t*)data_or_null(g_idx);
  args.perm = (const int32_t*)data_or_null(perm);
  args.b_bias = data_or_null(bias);
  args.global_scale = data_or_null(gscale);
  args.workspace = (int32_t*)workspace.mutable_data_ptr();
  args.workspace_len = workspace.numel();
  args.size_m = m;
  args.size_n = n;
  args.size_k = k;
  args.num_groups = groups;
}

Tensor dense_gemm(const Tensor& a, const Tensor* c_in, const Tensor& w, const Tensor* bias, const Tensor& scales, const Tensor* gscale,
                  const Tensor* zeros, const Tensor* g_idx, const Tensor* perm, const Tensor& workspace, int64_t q_type, int64_t size_m,
                  int64_t size_n, int64_t size_k, bool is_k_full, bool use_atomic_add, bool use_fp32_reduce, bool is_zp_float) {
  TORCH_CHECK(a.dim() == 2 && a.size(0) == size_m, "Shape mismatch: a.size(0) = ", a.size(0), ", size_m = ", size_m);
  TORCH_CHECK(a.size(1) == size_k, "Shape mismatch: a.size(1) = ", a.size(1), ", size_k = ", size_k);
  TORCH_CHECK(size_k % 16 == 0, "size_k = ", size_k, " is not divisible by tile_size = 16");
  TORCH_CHECK(w.dim() == 2 && size_k / 16 == w.size(0), "Shape mismatch: b_q_weight.size(0) = ", w.size(0), ", size_k = ", size_k,
              ", tile_size = 16");
  TORCH_CHECK(w.size(1) % 16 == 0, "b_q_weight.size(1) = ", w.size(1), " is not divisible by tile_size = 16");
  const int64_t pf = pack_factor(q_type);
  TORCH_CHECK(size_n == w.size(1) / 16 * pf, "Shape mismatch: b_q_weight.size(1) = ", w.size(1), ", size_n = ", size_n,
              ", pack_factor = ", pf);
  TORCH_CHECK(a.is_cuda(), "A is not on GPU");
  TORCH_CHECK(a.stride(1) == 1, "A.stride(1) is not 1");
  TORCH_CHECK(a.stride(0) % 8 == 0, "A.stride(0) must divisible by 8");
  TORCH_CHECK((uintptr_t)a.const_data_ptr() % 16 == 0, "A must aligned to 16 bytes");
  TORCH_CHECK(w.is_cuda() && w.is_contiguous(), "b_q_weight is not a contiguous GPU tensor");
  TORCH_CHECK(w.scalar_type() == at::kInt, "b_q_weight type is not kInt");
  TORCH_CHECK(scales.is_cuda() && scales.is_contiguous(), "b_scales is not a contiguous GPU tensor");
  TORCH_CHECK(scales.dim() == 2 && scales.size(1) == size_n, "b_scales dim 1 = ", scales.size(-1), " is not size_n = ", size_n);
  const int64_t groups = scales.size(0);
  check_scales(a, scales, q_type, size_k, groups, gscale, 1);
  TORCH_CHECK(workspace.is_cuda() && workspace.scalar_type() == at::kInt, "workspace must be an int32 GPU tensor");
  TORCH_CHECK((g_idx == nullptr) == (perm == nullptr), "Unexpected g_idx.size(-1) = ", g_idx ? g_idx->numel() : 0,
              " and perm.size(-1) = ", perm ? perm->numel() : 0);
  for (const auto& [name, t] : {std::pair<const char*, const Tensor*>{"g_idx", g_idx}, {"perm", perm}})
    if (t)
      TORCH_CHECK(t->is_cuda() && t->is_contiguous() && t->scalar_type() == at::kInt && t->numel() == size_k, name,
                  " must be a contiguous int32 [size_k] GPU tensor");
  if (zeros) {
    TORCH_CHECK(zeros->is_cuda() && zeros->is_contiguous(), "b_zeros is not a contiguous GPU tensor");
    TORCH_CHECK(zeros->dim() == 2, "b_zeros rank = ", zeros->dim(), " is not 2");
    TORCH_CHECK(zeros->size(0) == groups, "b_zeros dim 0 = ", zeros->size(0), " is not num_groups = ", groups);
    if (is_zp_float) {  // HQQ: fp16 zero points shaped and permuted like the scales (gptq_marlin.cu:866-887)
      TORCH_CHECK(a.scalar_type() == at::kHalf, "Computation type must be float16 (half) when using float zero points.");
      TORCH_CHECK(zeros->scalar_type() == a.scalar_type(), "b_zeros type is not the type of a");
      TORCH_CHECK(zeros->size(1) == size_n, "b_zeros dim 1 = ", zeros->size(1), " is not size_n = ", size_n);
    } else {
      TORCH_CHECK(zeros->scalar_type() == at::kInt, "b_zeros type is not kInt");
      TORCH_CHECK(zeros->size(1) == size_n / 8, "b_zeros dim 1 = ", zeros->size(1), " is not size_n / pack_factor = ", size_n / 8);
    }
  }
  TORCH_CHECK(!is_zp_float || zeros, "is_zp_float = True needs b_zeros");
  const int wtype = wtype_code(q_type, zeros != nullptr);
  if (bias)
    TORCH_CHECK(bias->is_cuda() && bias->numel() == size_n && bias->stride(-1) == 1 && bias->scalar_type() == a.scalar_type(),
                "b_bias.size(0) must be size_n, stride 1, dtype of a");
  Tensor c;
  if (c_in) {
    c = *c_in;
    TORCH_CHECK(c.is_cuda() && c.is_contiguous(), "c is not a contiguous GPU tensor");
    TORCH_CHECK(c.dim() == 2 && c.size(0) == size_m && c.size(1) == size_n && c.scalar_type() == a.scalar_type(), "Shape mismatch: c");
  } else {
    c = at::empty({size_m, size_n}, a.options());
  }
  if (size_m == 0) return c;
  const int flags = (use_fp32_reduce ? W4A16_F_USE_FP32_REDUCE : 0) | (is_k_full ? W4A16_F_IS_K_FULL : 0) |
                    (use_atomic_add ? W4A16_F_USE_ATOMIC_ADD : 0) | (is_zp_float ? W4A16_F_ZP_FLOAT : 0);
  w4a16_gemm_args args{};
  fill_common(args, a, c, w, bias, scales, zeros, g_idx, perm, gscale, workspace, wtype, size_m, size_n, size_k, groups, flags);
  run_gemm(args, a);
  return c;
}

// zero points are absent when their last dimension is empty, whatever the others are
const Tensor* present_zeros(const OptTensor& t) { return t.has_value() && t->defined() && t->size(-1) > 0 ? &*t : nullptr; }

Tensor gptq_marlin_gemm(const Tensor& a, const OptTensor& c_or_none, const Tensor& b_q_weight, const OptTensor& b_bias_or_none,
                        const Tensor& b_scales, const OptTensor& global_scale, const OptTensor& b_zeros_or_none,
                        const OptTensor& g_idx_or_none, const OptTensor& perm_or_none, const Tensor& workspace, int64_t b_q_type,
                        int64_t size_m, int64_t size_n, int64_t size_k, bool is_k_full, bool use_atomic_add, bool use_fp32_reduce,
                        bool is_zp_float) {
  return dense_gemm(a, c_or_none.has_value() ? &*c_or_none : nullptr, b_q_weight, present(b_bias_or_none), b_scales,
                    present(global_scale), present_zeros(b_zeros_or_none), present(g_idx_or_none), present(perm_or_none), workspace,
                    b_q_type, size_m, size_n, size_k, is_k_full, use_atomic_add, use_fp32_reduce, is_zp_float);
}

// One launch of the MoE GEMM.  silu_and_mul: c is [size_m * top_k, size_n / 2] = silu(gate) * up; sum_top_k > 0: c is
// [size_m * top_k / sum_top_k, size_n], already zero, and receives the sum of each token's rows; zero_fill: a tensor the
// launch clears on the side (the output of a later sum_top_k launch).
Tensor moe_gemm(const Tensor& a, const OptTensor& c_or_none, const Tensor& w, const OptTensor& bias_or_none, const Tensor& scales,
                const OptTensor& global_scale, const OptTensor& zeros_or_none, const OptTensor& g_idx_or_none,
                const OptTensor& perm_or_none, const Tensor& workspace, const Tensor& sorted_token_ids, const Tensor& expert_ids,
                const Tensor& num_tokens_past_padded, const Tensor& topk_weights, int64_t block, int64_t top_k,
                bool mul_topk_weights, int64_t q_type, int64_t size_m, int64_t size_n, int64_t size_k, bool is_full_k,
                bool use_atomic_add, bool use_fp32_reduce, bool is_zp_float, bool silu_and_mul, int64_t sum_top_k,
                const OptTensor& zero_fill) {
  TORCH_CHECK(a.is_cuda() && a.is_contiguous() && a.dim() == 2, "A is not a contiguous 2-D GPU tensor");
  TORCH_CHECK(a.size(0) == size_m, "Shape mismatch: a.size(0) = ", a.size(0), ", size_m = ", size_m);
  TORCH_CHECK(a.size(1) == size_k, "Shape mismatch: a.size(1) = ", a.size(1), ", size_k = ", size_k);
  TORCH_CHECK(block == 8 || (block % 16 == 0 && block >= 16 && block <= 64) || block == 128, "unsupported moe_block_size=", block);
  TORCH_CHECK(w.is_cuda() && w.is_contiguous() && w.dim() == 3 && w.scalar_type() == at::kInt,
              "b_q_weight is not a contiguous 3-D int32 GPU tensor");
  const int64_t experts = w.size(0);
  TORCH_CHECK(size_k % 16 == 0 && w.size(1) == size_k / 16, "Shape mismatch: b_q_weight.size(1) = ", w.size(1), ", size_k = ", size_k,
              ", tile_size = 16");
  const int64_t pf = pack_factor(q_type);
  TORCH_CHECK(w.size(2) % 16 == 0 && size_n == w.size(2) / 16 * pf, "Shape mismatch: b_q_weight.size(2) = ", w.size(2),
              ", size_n = ", size_n, ", pack_factor = ", pf);
  TORCH_CHECK(scales.is_cuda() && scales.is_contiguous() && scales.dim() == 3, "b_scales rank is not 3");
  TORCH_CHECK(scales.size(0) == experts && scales.size(2) == size_n, "b_scales dim 2 = ", scales.size(2), " is not size_n = ", size_n);
  TORCH_CHECK(!is_zp_float, "float zero points (HQQ) are not implemented for the MoE op by the gfx950 W4A16 library");
  const int64_t groups = scales.size(1);
  const Tensor* gscale = present(global_scale);
  check_scales(a, scales, q_type, size_k, groups, gscale, experts);
  const Tensor *g_idx = present(g_idx_or_none), *perm = present(perm_or_none);
  TORCH_CHECK((g_idx == nullptr) == (perm == nullptr), "g_idx and perm must both be given or both be empty");
  for (const auto& [name, t] : {std::pair<const char*, const Tensor*>{"g_idx", g_idx}, {"perm", perm}})
    if (t)
      TORCH_CHECK(t->is_cuda() && t->is_contiguous() && t->scalar_type() == at::kInt && t->dim() == 2 && t->size(0) == experts &&
                      t->size(1) == size_k,
                  name, " must be a contiguous int32 [E, size_k] GPU tensor");
  const Tensor* zeros = present_zeros(zeros_or_none);
  if (zeros) {
    TORCH_CHECK(zeros->is_cuda() && zeros->is_contiguous() && zeros->scalar_type() == at::kInt && zeros->dim() == 3,
                "b_zeros rank = ", zeros->dim(), " is not 3");
    TORCH_CHECK(zeros->size(0) == experts && zeros->size(1) == groups && zeros->size(2) == size_n / 8, "b_zeros shape mismatch");
  }
  const int wtype = wtype_code(q_type, zeros != nullptr);
  const Tensor* bias = present(bias_or_none);
  if (bias)
    TORCH_CHECK(bias->is_cuda() && bias->is_contiguous() && bias->dim() == 2 && bias->size(0) == experts && bias->size(1) == size_n &&
                    bias->scalar_type() == a.scalar_type(),
                "b_bias must be [E, size_n]");
  TORCH_CHECK(workspace.is_cuda() && workspace.scalar_type() == at::kInt, "workspace must be an int32 GPU tensor");
  check_gpu_i32(sorted_token_ids, "sorted_token_ids");
  check_gpu_i32(expert_ids, "expert_ids");
  check_gpu_i32(num_tokens_past_padded, "num_tokens_past_padded");
  TORCH_CHECK(expert_ids.numel() * block >= sorted_token_ids.numel() - block + 1, "expert_ids is too short for sorted_token_ids");
  TORCH_CHECK(topk_weights.is_cuda() && topk_weights.scalar_type() == at::kFloat && topk_weights.is_contiguous(),
              "topk_weights must be a contiguous fp32 GPU tensor");
  TORCH_CHECK(!mul_topk_weights || topk_weights.numel() >= size_m * top_k, "topk_weights holds ", topk_weights.numel(),
              " weights, the rows need ", size_m * top_k);
  const int64_t c_rows = size_m * top_k / (sum_top_k > 1 ? sum_top_k : 1), c_cols = silu_and_mul ? size_n / 2 : size_n;
  if (silu_and_mul)
    TORCH_CHECK(size_n % 128 == 0, "fused SiLU-and-mul: size_n = ", size_n, " must be 2 * d with d a multiple of 64");
  if (sum_top_k)
    TORCH_CHECK((sum_top_k == 1 || sum_top_k == 2) && (size_m * top_k) % sum_top_k == 0, "unsupported sum_top_k = ", sum_top_k);
  Tensor c;
  if (c_or_none.has_value()) {
    c = *c_or_none;
    TORCH_CHECK(c.is_cuda() && c.is_contiguous() && c.scalar_type() == a.scalar_type(), "c is not a contiguous GPU tensor");
    TORCH_CHECK(c.dim() == 2 && c.size(0) == c_rows && c.size(1) == c_cols, "Shape mismatch: c");
  } else {
    TORCH_CHECK(!sum_top_k, "the fused top-k sum accumulates into a caller-provided, zeroed c");
    c = at::empty({c_rows, c_cols}, a.options());
  }
  if (zero_fill.has_value())
    TORCH_CHECK(zero_fill->is_cuda() && zero_fill->is_contiguous() && (uintptr_t)zero_fill->const_data_ptr() % 16 == 0 &&
                    zero_fill->nbytes() % 16 == 0,
                "zero_fill must be a contiguous, 16-byte aligned GPU tensor of a multiple of 16 bytes");
  if (size_m == 0) {
    if (zero_fill.has_value()) zero_fill->zero_();
    return c;
  }
  const int flags = W4A16_F_MOE | (use_fp32_reduce ? W4A16_F_USE_FP32_REDUCE : 0) | (silu_and_mul ? W4A16_F_SILU_AND_MUL : 0) |
                    (sum_top_k ? W4A16_F_SUM_TOPK : 0) | (is_full_k ? W4A16_F_IS_K_FULL : 0) |
                    (use_atomic_add ? W4A16_F_USE_ATOMIC_ADD : 0) | (mul_topk_weights ? W4A16_F_MUL_TOPK_WEIGHTS : 0);
  w4a16_gemm_args args{};
  fill_common(args, a, c, w, bias, scales, zeros, g_idx, perm, gscale, workspace, wtype, size_m, size_n, size_k, groups, flags);
  args.sorted_token_ids = (const int32_t*)sorted_token_ids.const_data_ptr();
  args.expert_ids = (const int32_t*)expert_ids.const_data_ptr();
  args.num_tokens_past_padded = (const int32_t*)num_tokens_past_padded.const_data_ptr();
  args.topk_weights = (const float*)topk_weights.const_data_ptr();
  args.n_sorted = std::min<int64_t>(sorted_token_ids.numel(), expert_ids.numel() * block);
  args.moe_block_size = (int32_t)block;
  args.top_k = (int32_t)top_k;
  args.num_experts = (int32_t)experts;
  args.sum_top_k = (int32_t)sum_top_k;
  if (zero_fill.has_value()) {
    args.zero_fill = zero_fill->mutable_data_ptr();
    args.zero_fill_bytes = (int64_t)zero_fill->nbytes();
  }
  run_gemm(args, a);
  return c;
}

Tensor moe_wna16_marlin_gemm(const Tensor& a, const OptTensor& c_or_none, const Tensor& b_q_weight, const OptTensor& b_bias_or_none,
                             const Tensor& b_scales, const OptTensor& global_scale, const OptTensor& b_zeros_or_none,
                             const OptTensor& g_idx_or_none, const OptTensor& perm_or_none, const Tensor& workspace,
                             const Tensor& sorted_token_ids, const Tensor& expert_ids, const Tensor& num_tokens_past_padded,
                             const Tensor& topk_weights, int64_t moe_block_size, int64_t top_k, bool mul_topk_weights,
                             bool /*is_ep*/, int64_t b_q_type_id, int64_t size_m, int64_t size_n, int64_t size_k, bool is_full_k,
                             bool use_atomic_add, bool use_fp32_reduce, bool is_zp_float) {
  return moe_gemm(a, c_or_none, b_q_weight, b_bias_or_none, b_scales, global_scale, b_zeros_or_none, g_idx_or_none, perm_or_none,
                  workspace, sorted_token_ids, expert_ids, num_tokens_past_padded, topk_weights, moe_block_size, top_k,
                  mul_topk_weights, b_q_type_id, size_m, size_n, size_k, is_full_k, use_atomic_add, use_fp32_reduce, is_zp_float,
                  false, 0, std::nullopt);
}

void moe_marlin_gemm_fused(const Tensor& a, const Tensor& c, const Tensor& b_q_weight, const OptTensor& b_bias_or_none,
                           const Tensor& b_scales, const OptTensor& global_scale, const OptTensor& b_zeros_or_none,
                           const OptTensor& g_idx_or_none, const OptTensor& perm_or_none, const Tensor& workspace,
                           const Tensor& sorted_token_ids, const Tensor& expert_ids, const Tensor& num_tokens_past_padded,
                           const Tensor& topk_weights, int64_t moe_block_size, int64_t top_k, bool mul_topk_weights,
                           int64_t b_q_type_id, int64_t size_m, int64_t size_n, int64_t size_k, bool is_full_k, bool silu_and_mul,
                           int64_t sum_top_k, const OptTensor& zero_fill) {
  moe_gemm(a, c, b_q_weight, b_bias_or_none, b_scales, global_scale, b_zeros_or_none, g_idx_or_none, perm_or_none, workspace,
           sorted_token_ids, expert_ids, num_tokens_past_padded, topk_weights, moe_block_size, top_k, mul_topk_weights, b_q_type_id,
           size_m, size_n, size_k, is_full_k, false, true, false, silu_and_mul, sum_top_k, zero_fill);
}

// ---------------------------------------------------------------------------------------------------- MoE glue
void moe_align_block_size(const Tensor& topk_ids, int64_t num_experts, int64_t block_size, const Tensor& sorted_token_ids,
                          const Tensor& experts_ids, const Tensor& num_tokens_post_pad) {
  TORCH_CHECK(topk_ids.is_cuda() && topk_ids.is_contiguous(), "topk_ids must be a contiguous GPU tensor");
  const Tensor ids = topk_ids.scalar_type() == at::kInt ? topk_ids : topk_ids.to(at::kInt);
  for (const Tensor* t : {&sorted_token_ids, &experts_ids, &num_tokens_post_pad}) check_gpu_i32(*t, "outputs");
  OnDevice on(topk_ids);
  check_rc(w4a16_moe_align_block_size((const int32_t*)ids.const_data_ptr(), ids.numel(), (int32_t)num_experts, (int32_t)block_size,
                                      (int32_t*)sorted_token_ids.mutable_data_ptr(), sorted_token_ids.numel(),
                                      (int32_t*)experts_ids.mutable_data_ptr(), experts_ids.numel(),
                                      (int32_t*)num_tokens_post_pad.mutable_data_ptr(), stream_of(topk_ids)));
}

void batched_moe_align_block_size(int64_t max_tokens_per_batch, int64_t block_size, const Tensor& expert_num_tokens,
                                  const Tensor& sorted_token_ids, const Tensor& experts_ids, const Tensor& num_tokens_post_pad) {
  TORCH_CHECK(expert_num_tokens.is_cuda() && expert_num_tokens.is_contiguous() && expert_num_tokens.dim() == 1,
              "expert_num_tokens must be a contiguous 1-D GPU tensor");
  const Tensor n = expert_num_tokens.scalar_type() == at::kInt ? expert_num_tokens : expert_num_tokens.to(at::kInt);
  for (const Tensor* t : {&sorted_token_ids, &experts_ids, &num_tokens_post_pad}) check_gpu_i32(*t, "outputs");
  OnDevice on(n);
  check_rc(w4a16_batched_moe_align_block_size(max_tokens_per_batch, (int32_t)block_size, (const int32_t*)n.const_data_ptr(),
                                              (int32_t)n.numel(), (int32_t*)sorted_token_ids.mutable_data_ptr(),
                                              sorted_token_ids.numel(), (int32_t*)experts_ids.mutable_data_ptr(), experts_ids.numel(),
                                              (int32_t*)num_tokens_post_pad.mutable_data_ptr(), stream_of(n)));
}

void moe_sum(const Tensor& input, const Tensor& output) {
  TORCH_CHECK(input.is_cuda() && input.is_contiguous() && input.dim() == 3, "input must be a contiguous [T, topk, d] GPU tensor");
  TORCH_CHECK(output.is_cuda() && output.is_contiguous() && output.scalar_type() == input.scalar_type() && output.dim() == 2 &&
                  output.size(0) == input.size(0) && output.size(1) == input.size(2),
              "output must be a contiguous [T, d] GPU tensor");
  OnDevice on(input);
  check_rc(w4a16_moe_sum(input.const_data_ptr(), output.mutable_data_ptr(), input.size(0), (int32_t)input.size(1), input.size(2),
                         dtype_code(input.scalar_type()), stream_of(input)));
}

void silu_and_mul(const Tensor& result, const Tensor& input) {
  const int64_t d = input.size(-1) / 2;
  TORCH_CHECK(input.is_cuda() && result.is_cuda() && input.is_contiguous() && result.is_contiguous(),
              "tensors must be contiguous GPU tensors");
  TORCH_CHECK(result.size(-1) == d && result.numel() * 2 == input.numel() && result.scalar_type() == input.scalar_type(), "shape mismatch");
  OnDevice on(input);
  check_rc(w4a16_silu_and_mul(input.const_data_ptr(), result.mutable_data_ptr(), d ? input.numel() / (2 * d) : 0, d,
                              dtype_code(input.scalar_type()), stream_of(input)));
}

void topk_softmax(const Tensor& topk_weights, const Tensor& topk_indices, const Tensor& token_expert_indices,
                  const Tensor& gating_output, bool renormalize) {
  TORCH_CHECK(gating_output.is_cuda() && gating_output.is_contiguous() && gating_output.dim() == 2,
              "gating_output must be a contiguous [num_tokens, num_experts] GPU tensor");
  const int64_t tokens = gating_output.size(0), experts = gating_output.size(1), topk = topk_weights.size(-1);
  const auto shape_ok = [&](const Tensor& t) {
    return t.is_cuda() && t.is_contiguous() && t.dim() == 2 && t.size(0) == tokens && t.size(1) == topk;
  };
  TORCH_CHECK(topk_weights.scalar_type() == at::kFloat && shape_ok(topk_weights), "topk_weights must be fp32 [num_tokens, topk]");
  TORCH_CHECK(token_expert_indices.scalar_type() == at::kInt && shape_ok(token_expert_indices),
              "token_expert_indices must be int32 [num_tokens, topk]");
  TORCH_CHECK(shape_ok(topk_indices), "topk_indices shape mismatch");
  const auto t = gating_output.scalar_type();
  TORCH_CHECK(t == at::kHalf || t == at::kBFloat16 || t == at::kFloat, "gating_output must be fp16, bf16 or fp32");
  const int code = t == at::kHalf ? W4A16_DTYPE_F16 : t == at::kBFloat16 ? W4A16_DTYPE_BF16 : W4A16_DTYPE_F32;
  const bool direct = topk_indices.scalar_type() == at::kInt;
  const Tensor ids = direct ? topk_indices : at::empty({tokens, topk}, topk_indices.options().dtype(at::kInt));
  OnDevice on(gating_output);
  check_rc(w4a16_topk_softmax(gating_output.const_data_ptr(), code, (float*)topk_weights.mutable_data_ptr(),
                              (int32_t*)ids.mutable_data_ptr(), (int32_t*)token_expert_indices.mutable_data_ptr(), tokens,
                              (int32_t)experts, (int32_t)topk, renormalize ? 1 : 0, stream_of(gating_output)));
  if (!direct) topk_indices.copy_(ids);
}

// ------------------------------------------------------------------------------------------------ registration
using Registrar = void (*)(torch::Library&, const char*);
#define OP(fn) {#fn, [](torch::Library& lib, const char* name) { lib.impl(name, torch::CppFunction::makeFromUnboxedFunction(&fn)); }}
const std::pair<const char*, Registrar> kOps[] = {
    OP(gptq_marlin_gemm), OP(gptq_marlin_repack), OP(awq_marlin_repack), OP(permute_cols), OP(silu_and_mul),
    OP(moe_wna16_marlin_gemm), OP(moe_align_block_size), OP(batched_moe_align_block_size), OP(moe_sum), OP(topk_softmax),
    OP(moe_marlin_gemm_fused)};
#undef OP

// register_impl(namespace, name): attaches this file's implementation of `name` to the CUDA key of namespace::name
PyObject* py_register_impl(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  const char *ns, *name;
  if (!PyArg_ParseTuple(args, "ss", &ns, &name)) return nullptr;
  static std::vector<std::unique_ptr<torch::Library>> libs;  // (registrations live as long as their Library)
  for (const auto& [op, attach] : kOps)
    if (std::string(op) == name) {
      libs.push_back(std::make_unique<torch::Library>(torch::Library::IMPL, ns, c10::DispatchKey::CUDA, __FILE__, __LINE__));
      attach(*libs.back(), op);
      Py_RETURN_NONE;
    }
  PyErr_Format(PyExc_KeyError, "no native implementation of %s::%s", ns, name);
  return nullptr;
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------------------------------ direct eager entry
// Nothing but the CUDA kernel wants to see the call: no function or dispatch mode, tracer or profiler is on; the tensor is a
// Tensor or Parameter itself (a subclass with only __torch_function__ has the keys of a plain tensor, so its type is looked at),
// carries no key beyond an ordinary GPU tensor's and needs no gradient.
bool nobody_listens() {
  const uint64_t on = c10::impl::tls_local_dispatch_key_set().included_.raw_repr();
  return (on & ~c10::default_included_set.raw_repr()) == 0 && !at::hasCallbacks() && !at::impl::torch_function_mode_enabled();
}
bool plain(const Tensor& t) {
  static const uint64_t keys = (c10::DispatchKeySet(c10::DispatchKey::CUDA) | c10::autocast_dispatch_keyset |
                                c10::getAutogradRelatedKeySetFromBackend(c10::BackendComponent::CUDABit)).raw_repr();
  return (t.key_set().raw_repr() & ~keys) == 0 && t.is_cuda() && !(t.requires_grad() && at::GradMode::is_enabled());
}

// Flags and counts as Python's own bool and int.  The dispatcher also takes whatever has a truth value or an index (ints, numpy
// scalars, tensors); false leaves such a call to it, so that it means the same here as there.
bool read_flag(PyObject* o, bool* out) {
  *out = o == Py_True;
  return PyBool_Check(o);
}
bool read_int(PyObject* o, int64_t* out) {
  int overflow = 0;
  *out = PyLong_CheckExact(o) ? PyLong_AsLongLongAndOverflow(o, &overflow) : 0;
  return PyLong_CheckExact(o) && !overflow;
}

// linear(x, qweight, scales, zeros, g_idx, sort_indices, workspace, type_id, size_n, size_k, is_k_full, bias, use_fp32_reduce)
// -> [..., size_n], or None: not a call for this path.  zeros, g_idx, sort_indices and bias may be None or empty.
PyObject* py_linear(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(nargs == 13, "linear: 13 arguments");
  if (!nobody_listens()) Py_RETURN_NONE;
  const Tensor* t[8] = {};
  static const int at_arg[8] = {0, 1, 2, 3, 4, 5, 6, 11};
  for (int i = 0; i < 8; ++i) {
    PyObject* o = args[at_arg[i]];
    if (o == Py_None) continue;
    if (!THPVariable_CheckExact(o)) Py_RETURN_NONE;
    t[i] = &THPVariable_Unpack(o);
    if (!plain(*t[i])) Py_RETURN_NONE;
  }
  if (!t[0] || !t[1] || !t[2] || !t[6] || t[0]->dim() < 1) Py_RETURN_NONE;
  const auto some = [](const Tensor* x) { return x && x->numel() > 0 ? x : nullptr; };
  int64_t q_type, n, k;
  bool k_full, fp32_reduce;
  if (!read_int(args[7], &q_type) || !read_int(args[8], &n) || !read_int(args[9], &k) || !read_flag(args[10], &k_full) ||
      !read_flag(args[12], &fp32_reduce))
    Py_RETURN_NONE;
  const Tensor& x = *t[0];
  const Tensor* zeros = t[3] && t[3]->size(-1) > 0 ? t[3] : nullptr;
  Tensor y;
  {
    pybind11::gil_scoped_release nogil;
    const Tensor x2 = x.dim() == 2 ? x : x.reshape({-1, x.size(-1)});
    y = dense_gemm(x2, nullptr, *t[1], some(t[7]), *t[2], nullptr, zeros, some(t[4]), some(t[5]), *t[6], q_type, x2.size(0), n, k,
                   k_full, false, fp32_reduce, false);
    if (x.dim() != 2) {
      std::vector<int64_t> shape(x.sizes().begin(), x.sizes().end());
      shape.back() = n;
      y = y.reshape(shape);
    }
  }
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// The tensors at `at` (None -> null) unpacked, or false: something there is not for this path.
bool plain_args(PyObject* const* args, std::initializer_list<int> at, const Tensor** out) {
  for (const int i : at) {
    PyObject* o = args[i];
    if (o != Py_None) {
      if (!THPVariable_CheckExact(o)) return false;
      out[i] = &THPVariable_Unpack(o);
      if (!plain(*out[i])) return false;
    }
  }
  return true;
}

// topk(gating_output, topk, renormalize) -> (weights fp32, ids int32, source rows int32), each [tokens, topk], or None: not a call
// for this path.
PyObject* py_topk(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(nargs == 3, "topk: 3 arguments");
  const Tensor* t[1] = {};
  if (!nobody_listens() || !plain_args(args, {0}, t) || !t[0] || t[0]->dim() != 2 || !t[0]->is_contiguous()) Py_RETURN_NONE;
  int64_t topk;
  bool renormalize;
  if (!read_int(args[1], &topk) || !read_flag(args[2], &renormalize)) Py_RETURN_NONE;
  Tensor w, ids, rows;
  {
    pybind11::gil_scoped_release nogil;
    const auto i32 = t[0]->options().dtype(at::kInt);
    w = at::empty({t[0]->size(0), topk}, t[0]->options().dtype(at::kFloat));
    ids = at::empty({t[0]->size(0), topk}, i32);
    rows = at::empty({t[0]->size(0), topk}, i32);
    topk_softmax(w, ids, rows, *t[0], renormalize);
  }
  PyObject* out = PyTuple_New(3);
  if (!out) return nullptr;
  PyTuple_SET_ITEM(out, 0, THPVariable_Wrap(std::move(w)));
  PyTuple_SET_ITEM(out, 1, THPVariable_Wrap(std::move(ids)));
  PyTuple_SET_ITEM(out, 2, THPVariable_Wrap(std::move(rows)));
  return out;
  END_HANDLE_TH_ERRORS
}

// moe(x, w1, w2, bias1, bias2, scales1, scales2, zeros1, zeros2, gscale1, gscale2, g_idx1, g_idx2, sort1, sort2, topk_weights,
//     topk_ids, workspace, type_id, block, num_experts, weight_on_input, is_k_full) -> [M, K], or None: not a call for this path.
// The launches of fused_marlin_moe's Python (align, GEMM1 with SiLU-and-mul, GEMM2, the top-k sum) for its default arguments:
// a layer of small experts takes the GPU 30-60 us at a few tokens, those calls took the host 52-71 us, with the routing, from here 28-30.
PyObject* py_moe(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(nargs == 23, "moe: 23 arguments");
  const Tensor* t[18] = {};
  if (!nobody_listens() || !plain_args(args, {0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16, 17}, t)) Py_RETURN_NONE;
  for (const int i : {0, 1, 2, 5, 6, 15, 16, 17})
    if (!t[i]) Py_RETURN_NONE;
  const Tensor &x = *t[0], &w1 = *t[1], &w2 = *t[2], &tw = *t[15], &ids = *t[16];
  int64_t q_type, block, experts;
  bool weight_on_input, k_full;
  if (!read_int(args[18], &q_type) || !read_int(args[19], &block) || !read_int(args[20], &experts) ||
      !read_flag(args[21], &weight_on_input) || !read_flag(args[22], &k_full))
    Py_RETURN_NONE;
  if (x.dim() != 2 || w2.dim() != 3 || ids.dim() != 2 || ids.scalar_type() != at::kInt || !ids.is_contiguous()) Py_RETURN_NONE;
  const int64_t m = x.size(0), k = x.size(1), n = w2.size(1) * 16, topk = ids.size(1), slots = m * topk;
  if (m == 0 || topk < 1 || n % 64 != 0) Py_RETURN_NONE;  // (the fused activation pairs n-tiles of 64 columns)
  Tensor out;
  {
    pybind11::gil_scoped_release nogil;
    const auto i32 = ids.options();
    const auto opt = [&](int i) { return t[i] ? OptTensor(*t[i]) : OptTensor(); };
    const int64_t sorted_len = slots + experts * (block - 1);
    const Tensor sorted = at::empty({sorted_len}, i32), owners = at::empty({(sorted_len + block - 1) / block}, i32),
                 padded = at::empty({1}, i32);
    moe_align_block_size(ids, experts, block, sorted, owners, padded);
    const Tensor act = at::empty({slots, n}, x.options());
    out = at::empty({m, k}, x.options());
    const bool sum2 = topk == 2;
    moe_gemm(x, act, w1, opt(3), *t[5], opt(9), opt(7), opt(11), opt(13), *t[17], sorted, owners, padded, tw, block, topk,
             weight_on_input, q_type, m, 2 * n, k, k_full, false, true, false, true, 0, sum2 ? OptTensor(out) : OptTensor());
    const Tensor y = topk <= 2 ? out : at::empty({slots, k}, x.options());
    moe_gemm(act, y, w2, opt(4), *t[6], opt(10), opt(8), opt(12), opt(14), *t[17], sorted, owners, padded, tw, block, 1,
             !weight_on_input, q_type, slots, k, n, k_full, false, true, false, false, sum2 ? 2 : 0, std::nullopt);
    if (topk > 2) moe_sum(y.view({m, topk, k}), out);
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

PyMethodDef kMethods[] = {{"register_impl", py_register_impl, METH_VARARGS, "attach the native implementation of an operator"},
                          {"linear", (PyCFunction)(void*)py_linear, METH_FASTCALL, "direct eager W4A16 linear"},
                          {"topk", (PyCFunction)(void*)py_topk, METH_FASTCALL, "direct eager routing"},
                          {"moe", (PyCFunction)(void*)py_moe, METH_FASTCALL, "direct eager fused MoE layer"},
                          {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_torch_ops", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__torch_ops(void) { return PyModule_Create(&kModule); }
