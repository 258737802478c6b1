// MoE glue kernels for gfx950: token->expert block alignment, top-k sum, SiLU-and-mul.
//
// moe_align_block_size follows the contract of the reference op
// (vllm/model_executor/layers/fused_moe/moe_align_block_size.py:11-85, kernels
// csrc/moe/moe_align_sum_kernels.cu:83-268): sort the flattened (token, slot) indices by expert,
// pad every expert's run to a multiple of block_size with the value `numel`, emit one expert id
// per block (tail zero-filled) and the padded total.  Unlike the reference (atomic ranks, order
// inside an expert unspecified) the order here is stable — ascending flat index inside each
// expert — so the result is deterministic and equals the reference's torch golden
// (tests/kernels/moe/test_moe_align_block_size.py:92-168) element for element.
#include "gemm_common.h"

namespace w4a16 {

constexpr int ALIGN_THREADS = 1024;
constexpr int ALIGN_WAVES = ALIGN_THREADS / 64;
constexpr int ALIGN_MAX_EXPERTS = 1024;

// Up to 4 * ALIGN_THREADS * ALIGN_GROUPS ids: a workgroup holds all of them in its registers, every wavefront a contiguous run, asked for once.  Bound by
// its chain of round trips, which is cut to ids, histogram in LDS, positions and stores: a workgroup counts its own one to four experts in every run by
// ballots while the histogram fills, and every wavefront adds up the padded counts in front of them by itself (a scan by one wavefront stood behind
// a barrier of its own); the slots and blocks past the total are written by all workgroups.  The kernels that walked the ids two or three times: 333 ids of
// 128 experts 3.5 -> 2.8 us, 2000 6.0 -> 3.2, 4808 7.5 -> 4.1, 16384 of 64 8.7 -> 5.8, 65536 of 128 25.8 -> 14.9, 64000 of 8 26.4 -> 22.6
// (LDS atomics on eight addresses).
using i32x4 = int32_t __attribute__((ext_vector_type(4)));
constexpr int ALIGN_GROUPS = 16, ALIGN_OWN = 4;

// sum over the wavefront, in every lane (as wave_max below)
template <int CTRL>
__device__ __forceinline__ int dpp_add(int x) { return x + __builtin_amdgcn_update_dpp(0, x, CTRL, 0xf, 0xf, true); }
__device__ __forceinline__ int wave_sum(int x) {
  x = dpp_add<0x111>(x);  // row_shr:1, 2, 4, 8
  x = dpp_add<0x112>(x);
  x = dpp_add<0x114>(x);
  x = dpp_add<0x118>(x);
  x = dpp_add<0x142>(x);  // row_bcast:15
  x = dpp_add<0x143>(x);  // row_bcast:31
  return __builtin_amdgcn_readlane(x, 63);
}

template <int THREADS, int R>
__global__ __launch_bounds__(THREADS) void moe_align_held_kernel(
    const int32_t* __restrict__ topk_ids, int numel, int num_experts, int block_size, int vec, int32_t* __restrict__ sorted_ids, int sorted_len,
    int32_t* __restrict__ expert_ids, int expert_ids_len, int32_t* __restrict__ num_post_pad) {
  constexpr int WAVES = THREADS / 64;
  __shared__ int cnt[ALIGN_MAX_EXPERTS];
  __shared__ int run_cnt[ALIGN_OWN][WAVES];
  const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
  // ids of this lane: four consecutive ones of each of R groups; -1 past the end
  i32x4 v[R];
  const int i0 = (wv * R * 64 + lane) * 4;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = i0 + r * 256;
    if (vec && i + 4 <= numel) {
      v[r] = *(const i32x4*)(topk_ids + i);
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) v[r][q] = i + q < numel ? topk_ids[i + q] : -1;
    }
  }
  for (int e = t; e < num_experts; e += THREADS) cnt[e] = 0;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if ((unsigned)v[r][q] < (unsigned)num_experts) atomicAdd(&cnt[v[r][q]], 1);
  // this workgroup's experts: blockIdx.x, + gridDim.x, ... (at most ALIGN_OWN: host)
#pragma unroll
  for (int o = 0; o < ALIGN_OWN; ++o) {
    const int e = blockIdx.x + o * gridDim.x;
    if (e >= num_experts) break;
    int n = 0;
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int q = 0; q < 4; ++q) n += __popcll(__ballot(v[r][q] == e));
    if (lane == 0) run_cnt[o][wv] = n;
  }
  __syncthreads();
  auto padded = [&](int n) { return (n + block_size - 1) / block_size * block_size; };
  int before[ALIGN_OWN] = {}, all = 0;  // padded slots of the experts in front of each of this workgroup's, and of all
  for (int e = lane; e < num_experts; e += 64) {
    const int n = padded(cnt[e]);
    all += n;
#pragma unroll
    for (int o = 0; o < ALIGN_OWN; ++o) before[o] += e < (int)(blockIdx.x + o * gridDim.x) ? n : 0;
  }
  const int total = wave_sum(all);
#pragma unroll
  for (int o = 0; o < ALIGN_OWN; ++o) {
    const int e = blockIdx.x + o * gridDim.x;
    if (e >= num_experts) break;
    const int off = wave_sum(before[o]), n = cnt[e], end = off + padded(n);
    int pos = off + wave_sum(lane < wv ? run_cnt[o][lane] : 0);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      unsigned long long m[4];
      int in_front = 0, hits = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        m[q] = __ballot(v[r][q] == e);
        in_front += __builtin_amdgcn_mbcnt_hi((uint32_t)(m[q] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m[q], 0));
        hits += __popcll(m[q]);
      }
      if (hits) {
        int p = pos + in_front;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if (v[r][q] == e) {
            if (p < sorted_len) sorted_ids[p] = i0 + r * 256 + q;
            ++p;
          }
        }
      }
      pos += hits;
    }
    for (int i = off + n + t; i < end && i < sorted_len; i += THREADS) sorted_ids[i] = numel;
    const int b1 = end / block_size;
    for (int b = off / block_size + t; b < b1 && b < expert_ids_len; b += THREADS) expert_ids[b] = e;
  }
  // slots past the total hold numel, blocks past it 0
  const int at = blockIdx.x * THREADS + t, step = gridDim.x * THREADS;
  for (int i = total + at; i < sorted_len; i += step) sorted_ids[i] = numel;
  for (int b = total / block_size + at; b < expert_ids_len; b += step) expert_ids[b] = 0;
  if (at == 0) *num_post_pad = total;
}

// The same contract for longer id lists:
//   * every thread fetches its ids with 16-byte loads, several in flight, for the histogram (LDS atomics: per-expert
//     ballot counts for the few-expert case, where lanes queue on a few addresses, measured slower);
//   * the ids of an expert are placed by `spe` wavefronts of a workgroup, each on a contiguous slice of the ids:
//     count the matches of the slice, exchange the counts through LDS, place from the slice's start position.  A lane
//     holds four consecutive ids; a match's rank is the matches of the lanes in front plus its own earlier components,
//     so the order inside an expert stays the order of the ids (stable, deterministic).
constexpr int ALIGN_ROUND = 8;  // 16-byte loads in flight per lane in the placement passes (2048 ids per wavefront round)
template <bool VEC>  // topk_ids on 16 bytes
__global__ __launch_bounds__(ALIGN_THREADS) void moe_align_sliced_kernel(
    const int32_t* __restrict__ topk_ids, int numel, int num_experts, int block_size, int spe,
    int32_t* __restrict__ sorted_ids, int sorted_len, int32_t* __restrict__ expert_ids, int expert_ids_len,
    int32_t* __restrict__ num_post_pad) {
  __shared__ int cnt[ALIGN_MAX_EXPERTS];
  __shared__ int off[ALIGN_MAX_EXPERTS + 1];
  __shared__ int slice_cnt[ALIGN_WAVES];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const unsigned long long lt = (1ull << lane) - 1ull;
  for (int e = t; e < num_experts; e += ALIGN_THREADS) cnt[e] = 0;
  __syncthreads();
  const int nvec = numel >> 2;  // whole 16-byte groups; the last numel & 3 ids are handled one by one
  auto load4 = [&](int vi) {
    if constexpr (VEC) return ((const i32x4*)topk_ids)[vi];
    const int32_t* at = topk_ids + 4 * vi;
    return i32x4{at[0], at[1], at[2], at[3]};
  };

  // ---- histogram
  for (int v0 = 0; v0 < nvec; v0 += 4 * ALIGN_THREADS) {
    i32x4 v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int vi = v0 + j * ALIGN_THREADS + t;
      v[j] = vi < nvec ? load4(vi) : i32x4{-1, -1, -1, -1};
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int e = v[j][q];
        if (e >= 0 && e < num_experts) atomicAdd(&cnt[e], 1);
      }
    }
  }
  if (t < (numel & 3)) {
    const int e = topk_ids[4 * nvec + t];
    if (e >= 0 && e < num_experts) atomicAdd(&cnt[e], 1);
  }
  __syncthreads();
  if (t < 64) {  // wave 0: exclusive scan of padded counts, 64 experts per round
    int acc = 0;
    for (int base = 0; base < num_experts; base += 64) {
      const int e = base + t;
      const int padded = e < num_experts ? (cnt[e] + block_size - 1) / block_size * block_size : 0;
      int incl = padded;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int v = __shfl_up(incl, d, 64);
        if (t >= d) incl += v;
      }
      if (e < num_experts) off[e] = acc + incl - padded;
      acc += __shfl(incl, 63, 64);
    }
    if (t == 0) off[num_experts] = acc;
  }
  __syncthreads();
  const int total = off[num_experts];
  if (blockIdx.x == 0) {
    if (t == 0) *num_post_pad = total;
    // expert id of every block; blocks past the padded total are zero-filled; slots past the total hold numel
    for (int e = t; e < num_experts; e += ALIGN_THREADS) {
      const int b0 = off[e] / block_size, b1 = off[e + 1] / block_size;
      for (int b = b0; b < b1 && b < expert_ids_len; ++b) expert_ids[b] = e;
    }
    for (int b = total / block_size + t; b < expert_ids_len; b += ALIGN_THREADS) expert_ids[b] = 0;
    for (int i = total + t; i < sorted_len; i += ALIGN_THREADS) sorted_ids[i] = numel;
  }

  // ---- placement: workgroup turn `eg` handles experts eg * epw .. + epw - 1, `spe` wavefronts each
  const int epw = ALIGN_WAVES / spe;
  const int j = wv / spe, sl = wv % spe;
  // slice of the 16-byte groups: whole wavefront loads (64 groups)
  const int per = ((nvec + spe - 1) / spe + 63) / 64 * 64;
  const int vb = min(sl * per, nvec), ve = min(vb + per, nvec);
  for (int eg = blockIdx.x; eg * epw < num_experts; eg += gridDim.x) {
    const int e = eg * epw + j;
    const bool live = e < num_experts && cnt[e] > 0;
    // matches of expert e in groups [vb, ve): pass 0 counts, pass 1 places from `pos`
    int pos = 0;
    for (int pass = 0; pass < 2; ++pass) {
      int seen = 0;
      if (live) {
        for (int v0 = vb; v0 < ve; v0 += 64 * ALIGN_ROUND) {
          i32x4 v[ALIGN_ROUND];
#pragma unroll
          for (int r = 0; r < ALIGN_ROUND; ++r) {
            const int vi = v0 + 64 * r + lane;
            v[r] = vi < ve ? load4(vi) : i32x4{-1, -1, -1, -1};
          }
#pragma unroll
          for (int r = 0; r < ALIGN_ROUND; ++r) {
            unsigned long long m[4];
            int before = 0, all = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              m[q] = __ballot(v[r][q] == e);
              before += __popcll(m[q] & lt);
              all += __popcll(m[q]);
            }
            if (pass == 1 && all) {
              int p = pos + seen + before;
              const int idx = 4 * (v0 + 64 * r + lane);
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                if (v[r][q] == e) {
                  if (p < sorted_len) sorted_ids[p] = idx + q;
                  ++p;
                }
              }
            }
            seen += all;
          }
        }
        // the last slice also owns the numel & 3 ids past the 16-byte groups
        if (sl == spe - 1) {
          const int i = 4 * nvec + lane;
          const bool hit = lane < (numel & 3) && topk_ids[i] == e;
          const unsigned long long m = __ballot(hit);
          if (pass == 1 && hit) {
            const int p = pos + seen + __popcll(m & lt);
            if (p < sorted_len) sorted_ids[p] = i;
          }
          seen += __popcll(m);
        }
      }
      if (pass == 0) {
        if (lane == 0) slice_cnt[wv] = seen;
        __syncthreads();
        if (live) {
          pos = off[e];
          for (int s2 = 0; s2 < sl; ++s2) pos += slice_cnt[j * spe + s2];
        }
        __syncthreads();  // slice_cnt is rewritten in the next turn
      }
    }
    // padding slots of the expert: by its first slice's wavefront
    if (e < num_experts && sl == 0) {
      const int padded = (cnt[e] + block_size - 1) / block_size * block_size;
      for (int i = off[e] + cnt[e] + lane; i < off[e] + padded && i < sorted_len; i += 64) sorted_ids[i] = numel;
    }
  }
}

// B terms' loads in flight together (a few tokens give too few wavefronts to hide one round trip per term); added in
// term order
template <int DT, int B>
__device__ __forceinline__ void moe_sum_terms(const uint16_t* __restrict__ in, int64_t tok, int top_k, int64_t hidden8,
                                              int64_t col, float* acc) {
  for (int k0 = 0; k0 < top_k; k0 += B) {
    u32x4 v[B];
#pragma unroll
    for (int i = 0; i < B; ++i)
      v[i] = *(const u32x4*)(in + ((tok * top_k + min(k0 + i, top_k - 1)) * hidden8 + col) * 8);
#pragma unroll
    for (int i = 0; i < B; ++i) {
      if (k0 + i < top_k) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          acc[2 * j] += DT == DT_F16 ? f16_lo_f32(v[i][j]) : bf16_lo_f32(v[i][j]);
          acc[2 * j + 1] += DT == DT_F16 ? f16_hi_f32(v[i][j]) : bf16_hi_f32(v[i][j]);
        }
      }
    }
  }
}

template <int DT>
__global__ __launch_bounds__(256) void moe_sum_kernel(const uint16_t* __restrict__ in, uint16_t* __restrict__ out,
                                                      int64_t total8, int top_k, int64_t hidden8) {
  // one thread per 8 consecutive output elements
  for (int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x; idx < total8; idx += (int64_t)gridDim.x * 256) {
    const int64_t tok = idx / hidden8, col = idx % hidden8;
    float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (top_k <= 2)
      moe_sum_terms<DT, 2>(in, tok, top_k, hidden8, col, acc);
    else if (top_k <= 4)
      moe_sum_terms<DT, 4>(in, tok, top_k, hidden8, col, acc);
    else
      moe_sum_terms<DT, 8>(in, tok, top_k, hidden8, col, acc);
    u32x4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      o[j] = DT == DT_F16 ? pack_f16(acc[2 * j], acc[2 * j + 1]) : pack_bf16(acc[2 * j], acc[2 * j + 1]);
    *(u32x4*)(out + idx * 8) = o;
  }
}

// out = T(silu_f32(x)) * y evaluated like the reference's act_and_mul_kernel<silu>
// (csrc/activation_kernels.cu:22-40): SiLU in fp32 rounded to T, then one multiply rounded to T.
template <int DT>
__global__ __launch_bounds__(256) void silu_and_mul_kernel(const uint16_t* __restrict__ in,
                                                           uint16_t* __restrict__ out, int64_t total8,
                                                           int64_t d8) {
  for (int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x; idx < total8; idx += (int64_t)gridDim.x * 256) {
    const int64_t tok = idx / d8, col = idx % d8;
    const u32x4 x = *(const u32x4*)(in + (tok * 2 * d8 + col) * 8);
    const u32x4 y = *(const u32x4*)(in + (tok * 2 * d8 + d8 + col) * 8);
    u32x4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float xv[2], yv[2], r[2];
      xv[0] = DT == DT_F16 ? f16_lo_f32(x[j]) : bf16_lo_f32(x[j]);
      xv[1] = DT == DT_F16 ? f16_hi_f32(x[j]) : bf16_hi_f32(x[j]);
      yv[0] = DT == DT_F16 ? f16_lo_f32(y[j]) : bf16_lo_f32(y[j]);
      yv[1] = DT == DT_F16 ? f16_hi_f32(y[j]) : bf16_hi_f32(y[j]);
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const float s = silu_f32(xv[q]);
        const uint32_t sr = DT == DT_F16 ? pack_f16(s, 0.f) : pack_bf16(s, 0.f);
        const float st = DT == DT_F16 ? f16_lo_f32(sr) : bf16_lo_f32(sr);
        r[q] = st * yv[q];
      }
      o[j] = DT == DT_F16 ? pack_f16(r[0], r[1]) : pack_bf16(r[0], r[1]);
    }
    *(u32x4*)(out + idx * 8) = o;
  }
}


// Routing: fp32 softmax over the experts of one token, then top-k by repeated arg-max (ties -> lowest expert
// index), as the reference's topk_softmax (csrc/moe/topk_softmax_kernels.cu:127-211, 676-705):
// weights are the softmax probabilities of the chosen experts, optionally renormalised to sum to 1
// (a zero sum divides by 1); token_expert_indices[t, k] = k * num_tokens + t.
// One wavefront per token; lane l holds experts l, l + 64, ... (PL of them: 1, 2 or 4 up to 64, 128 or 256 experts, 16 above) in
// registers.  A pick is a maximum over the wavefront by DPP moves (no LDS crossbar), then one ballot per register from the lowest
// expert numbers up: the lowest index among equals.  Lane k keeps pick k; weights are rescaled and written once, at the end.
// Bound by latency (a chain of topk maxima); with 16 registers per lane whatever the expert count, two-operand butterflies through
// the crossbar and the rescaling read back from memory it took 13.0 us on 601 tokens x 128 experts, top-8, now 5.0.
constexpr int TOPK_PER_LANE = 16;  // up to 1024 experts

template <typename T>
__device__ __forceinline__ float gate_to_f32(T v);
template <>
__device__ __forceinline__ float gate_to_f32<float>(float v) { return v; }
template <>
__device__ __forceinline__ float gate_to_f32<_Float16>(_Float16 v) { return (float)v; }
template <>
__device__ __forceinline__ float gate_to_f32<__bf16>(__bf16 v) { return (float)v; }

// maximum over the wavefront, in every lane (DPP: row shifts within 16 lanes, then row broadcasts; the last lane has it)
template <int CTRL>
__device__ __forceinline__ float dpp_max(float x) {
  const int v = __builtin_bit_cast(int, x);
  return fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false)));
}
__device__ __forceinline__ float wave_max(float x) {
  x = dpp_max<0x111>(x);  // row_shr:1
  x = dpp_max<0x112>(x);
  x = dpp_max<0x114>(x);
  x = dpp_max<0x118>(x);
  x = dpp_max<0x142>(x);  // row_bcast:15
  x = dpp_max<0x143>(x);  // row_bcast:31
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), 63));
}

// the same of whole numbers: one instruction a step (a lane that has no source reads the lowest number)
template <int CTRL>
__device__ __forceinline__ int dpp_imax(int x) { return max(x, __builtin_amdgcn_update_dpp((int)0x80000000, x, CTRL, 0xf, 0xf, false)); }
__device__ __forceinline__ int wave_imax(int x) {
  x = dpp_imax<0x111>(x);
  x = dpp_imax<0x112>(x);
  x = dpp_imax<0x114>(x);
  x = dpp_imax<0x118>(x);
  x = dpp_imax<0x142>(x);
  x = dpp_imax<0x143>(x);
  return __builtin_amdgcn_readlane(x, 63);
}
// sum over the wavefront, in every lane, pairs 32, 16, ... 1 lanes apart (rotations by 8, 4, 2 and 1 in rows of 16 meet the lane that far apart, or one
// with the same sum)
template <int CTRL>
__device__ __forceinline__ float dpp_rot_add(float x) {
  const int v = __builtin_bit_cast(int, x);
  return x + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float wave_sum_pairs(float x) {
  auto a = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(int, x), __builtin_bit_cast(int, x), false, false);
  x = __builtin_bit_cast(float, (int)a[0]) + __builtin_bit_cast(float, (int)a[1]);
  a = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(int, x), __builtin_bit_cast(int, x), false, false);
  x = __builtin_bit_cast(float, (int)a[0]) + __builtin_bit_cast(float, (int)a[1]);
  x = dpp_rot_add<0x128>(x);  // row_ror:8, 4, 2, 1
  x = dpp_rot_add<0x124>(x);
  x = dpp_rot_add<0x122>(x);
  return dpp_rot_add<0x121>(x);
}

// One wavefront per token.  Bound by its chain of dependent instructions: maximum, sum and, per pick, the largest probability and the first lane that holds
// it.  So the picks compare the probabilities as whole numbers (not negative: the same order; a step of the maximum is one instruction instead of three),
// the sum stays in the registers, and the loop over the picks has no branch (601 tokens of 128 experts, top-8 3.8 -> 2.9 us, 4096 tokens 5.5 -> 3.9,
// 1000 of 256 experts, top-16 6.9 -> 5.0, 16 of 8, top-2 2.3 -> 1.9; the same bits).
template <typename T, int PL>
__global__ __launch_bounds__(256) void topk_softmax_kernel(const T* __restrict__ gating, float* __restrict__ weights,
                                                           int32_t* __restrict__ ids, int32_t* __restrict__ src_rows,
                                                           int num_tokens, int num_experts, int topk, int renormalize) {
  const int lane = threadIdx.x & 63;
  const int tok = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (tok >= num_tokens) return;
  const T* row = gating + (int64_t)tok * num_experts;
  float v[PL];
  float mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < PL; ++i) {
    const int e = lane + 64 * i;
    v[i] = e < num_experts ? gate_to_f32<T>(row[e]) : -INFINITY;
    mx = fmaxf(mx, v[i]);
  }
  mx = wave_max(mx);
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < PL; ++i) {
    const int e = lane + 64 * i;
    v[i] = e < num_experts ? expf(v[i] - mx) : 0.f;
    sum += v[i];
  }
  sum = wave_sum_pairs(sum);
  // A row with a NaN or +inf (or nothing but -inf) has no probabilities: every sum of exponentials but that is 1 or more.  It
  // picks experts 0, 1, ... with NaN weights, so that its token's result is NaN and no id is out of range.
  const bool bad = !(sum > 0.f);
  int pr[PL];  // the probabilities' bits
#pragma unroll
  for (int i = 0; i < PL; ++i) {
    const int e = lane + 64 * i;
    pr[i] = __builtin_bit_cast(int, e < num_experts ? fmaxf(v[i] / sum, 0.f) : -1.f);  // (0 for a NaN) probabilities are >= 0: -1 marks "not a candidate"
  }
  const int64_t base = (int64_t)tok * topk;
  float selected = 0.f, my_w = 0.f;
  int my_e = 0;
  auto pick = [&](int k) {
    int top = pr[0];
#pragma unroll
    for (int i = 1; i < PL; ++i) top = max(top, pr[i]);
    top = wave_imax(top);  // (>= 0: topk <= num_experts)
    const float best = __builtin_bit_cast(float, top);
    int be = 0x7fffffff;
#pragma unroll
    for (int i = PL - 1; i >= 0; --i) {
      const unsigned long long m = __ballot(pr[i] == top);
      be = m ? 64 * i + __builtin_ctzll(m) : be;
    }
    selected += best;
    const bool mine = (k & 63) == lane;
    my_w = mine ? best : my_w;
    my_e = mine ? be : my_e;
#pragma unroll
    for (int i = 0; i < PL; ++i) pr[i] = lane + 64 * i == be ? __builtin_bit_cast(int, -1.f) : pr[i];
  };
  if (topk <= 64) {
    for (int k = 0; k < topk; ++k) pick(k);
  } else {
    for (int k = 0; k < topk; ++k) {
      pick(k);
      if ((k & 63) == lane) {  // more picks than lanes: kept in memory, each by the lane that rescales it
        weights[base + k] = bad ? __builtin_nanf("") : my_w;
        ids[base + k] = my_e;
        src_rows[base + k] = k * num_tokens + tok;
      }
    }
  }
  if (bad) my_w = __builtin_nanf("");
  const float denom = renormalize && selected > 0.f ? selected : 1.f;
  if (topk <= 64) {
    if (lane < topk) {
      weights[base + lane] = renormalize ? my_w / denom : my_w;
      ids[base + lane] = my_e;
      src_rows[base + lane] = lane * num_tokens + tok;
    }
  } else if (renormalize) {
    for (int k = lane; k < topk; k += 64) weights[base + k] /= denom;
  }
}

template <typename T>
static void launch_topk(const void* gating, float* weights, int32_t* ids, int32_t* src_rows, int64_t num_tokens, int num_experts,
                        int topk, int renormalize, hipStream_t st) {
  const int pl = num_experts <= 64 ? 1 : num_experts <= 128 ? 2 : num_experts <= 256 ? 4 : TOPK_PER_LANE;
  auto* fn = pl == 1 ? topk_softmax_kernel<T, 1> : pl == 2 ? topk_softmax_kernel<T, 2>
             : pl == 4 ? topk_softmax_kernel<T, 4> : topk_softmax_kernel<T, TOPK_PER_LANE>;
  hipLaunchKernelGGL(fn, dim3((unsigned)ceil_div(num_tokens, 4)), dim3(256), 0, st, (const T*)gating, weights, ids, src_rows,
                     (int)num_tokens, num_experts, topk, renormalize);
}

}  // namespace w4a16

using namespace w4a16;

// Alignment for activations already batched per expert ([B, max_tokens, K], batch_num_tokens[b] valid rows in batch
// b), the contract of the reference's batched_moe_align_block_size (csrc/moe/moe_align_sum_kernels.cu:18-80, 348-373):
// batch b's rows b * max_tokens + j, j < n_b, padded to a multiple of block_size with the value B * max_tokens, runs
// packed in batch order; one batch id per block, -1 past the last; the padded total.  One workgroup: an inclusive scan
// of the padded counts in LDS, then every output slot is written exactly once (its batch found by bisection).
__global__ __launch_bounds__(ALIGN_THREADS) void batched_moe_align_kernel(
    int num_batches, int max_tokens, int block_size, const int32_t* __restrict__ batch_num_tokens,
    int32_t* __restrict__ sorted_ids, int sorted_len, int32_t* __restrict__ block_ids, int32_t* __restrict__ num_post_pad) {
  __shared__ int incl[ALIGN_MAX_EXPERTS];  // inclusive scan of padded counts
  __shared__ int cnt[ALIGN_MAX_EXPERTS];
  const int t = threadIdx.x;
  const int n = t < num_batches ? min(max(batch_num_tokens[t], 0), max_tokens) : 0;
  cnt[t] = n;
  incl[t] = (n + block_size - 1) / block_size * block_size;
  __syncthreads();
  for (int d = 1; d < ALIGN_THREADS; d <<= 1) {
    const int add = t >= d ? incl[t - d] : 0;
    __syncthreads();
    incl[t] += add;
    __syncthreads();
  }
  const int total = incl[ALIGN_THREADS - 1];
  if (t == 0) *num_post_pad = total;
  const int sentinel = num_batches * max_tokens;
  auto batch_of = [&](int pos) {  // first b with incl[b] > pos (pos < total)
    int lo = 0, hi = num_batches - 1;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (incl[mid] > pos) hi = mid; else lo = mid + 1;
    }
    return lo;
  };
  for (int i = t; i < sorted_len; i += ALIGN_THREADS) {
    int v = sentinel;
    if (i < total) {
      const int b = batch_of(i);
      const int start = b == 0 ? 0 : incl[b - 1];
      if (i - start < cnt[b]) v = b * max_tokens + (i - start);
    }
    sorted_ids[i] = v;
  }
  for (int i = t; i < sorted_len / block_size; i += ALIGN_THREADS)
    block_ids[i] = i * block_size < total ? batch_of(i * block_size) : -1;
}

extern "C" int w4a16_moe_align_block_size(const int32_t* topk_ids, int64_t numel, int32_t num_experts,
                                          int32_t block_size, int32_t* sorted_token_ids, int64_t sorted_len,
                                          int32_t* expert_ids, int64_t expert_ids_len,
                                          int32_t* num_tokens_post_pad, void* stream) {
  W4A16_CHECK(topk_ids && sorted_token_ids && expert_ids && num_tokens_post_pad, "null pointer");
  W4A16_CHECK(num_experts >= 1 && num_experts <= ALIGN_MAX_EXPERTS, "num_experts = %d must be in [1, %d]",
              num_experts, ALIGN_MAX_EXPERTS);
  W4A16_CHECK(block_size >= 1, "block_size must be positive");
  W4A16_CHECK(numel >= 0 && numel < (1LL << 30), "bad topk_ids.numel()");
  W4A16_CHECK(sorted_len >= numel, "sorted_token_ids is shorter than topk_ids");
  const int vec = ((uintptr_t)topk_ids & 15) == 0;
  if (numel <= 4 * ALIGN_THREADS * ALIGN_GROUPS) {
    const int grid = num_experts < 256 ? num_experts : 256;
    // (256 threads start 1 us sooner than 1024: 2000 ids 3.2 us against 3.5; 4808 and 8192 ids 4.1 and 4.9 with 1024, 4.2 and 4.8 with 512)
    const int threads = numel <= 2048 ? 256 : ALIGN_THREADS;
    const int64_t r = ceil_div(numel, 4 * threads);  // groups per thread
    const auto fn = threads == 256 ? (r <= 1 ? moe_align_held_kernel<256, 1> : moe_align_held_kernel<256, 2>)
                    : r <= 1       ? moe_align_held_kernel<ALIGN_THREADS, 1>
                    : r <= 2       ? moe_align_held_kernel<ALIGN_THREADS, 2>
                    : r <= 4       ? moe_align_held_kernel<ALIGN_THREADS, 4>
                    : r <= 8       ? moe_align_held_kernel<ALIGN_THREADS, 8>
                                   : moe_align_held_kernel<ALIGN_THREADS, ALIGN_GROUPS>;
    fn<<<grid, threads, 0, (hipStream_t)stream>>>(topk_ids, (int)numel, num_experts, block_size, vec, sorted_token_ids, (int)sorted_len, expert_ids,
                                                  (int)expert_ids_len, num_tokens_post_pad);
    W4A16_HIP(hipGetLastError());
    return 0;
  }
  // slices per expert: enough wavefronts for 64 and more workgroups
  int spe = 1;
  while (spe < ALIGN_WAVES && num_experts * spe < 1024) spe *= 2;
  const int64_t turns = ceil_div(num_experts, ALIGN_WAVES / spe);
  const int grid = (int)(turns < 256 ? turns : 256);
  const auto fn = vec ? moe_align_sliced_kernel<true> : moe_align_sliced_kernel<false>;
  fn<<<grid, ALIGN_THREADS, 0, (hipStream_t)stream>>>(topk_ids, (int)numel, num_experts, block_size, spe, sorted_token_ids, (int)sorted_len, expert_ids,
                                                      (int)expert_ids_len, num_tokens_post_pad);
  W4A16_HIP(hipGetLastError());
  return 0;
}

// MoE act-order gather in front of the GEMM (the role of the reference's permute_cols_kernel<moe_block_size>,
// csrc/moe/marlin_moe_wna16/ops.cu:75-149): out[slot, k] = a[sorted_ids[slot] / top_k, perm_e[k]] for every valid slot,
// perm_e = the column order of the expert that owns the slot's block.  One workgroup per slot and turn: the source row is
// staged in LDS with 16-byte loads, every thread assembles 16-byte pieces of the output row from eight 2-byte LDS reads.
// Slots past the padded total, padding slots and blocks of experts of other ranks are skipped (their rows of `out` stay
// as they are: the GEMM kernels never store results of such rows).
namespace w4a16 {
constexpr int MG_MAX_K = 32768;  // 64 KB of LDS
template <bool STAGED>
__global__ __launch_bounds__(256) void moe_gather_rows_kernel(const uint16_t* __restrict__ a, int64_t lda,
                                                             const int32_t* __restrict__ perm,
                                                             const int32_t* __restrict__ sorted_ids,
                                                             const int32_t* __restrict__ expert_ids,
                                                             const int32_t* __restrict__ ntpp, int n_sorted, int block,
                                                             int top_k, int c_rows, int size_k,
                                                             uint16_t* __restrict__ out) {
  extern __shared__ __align__(16) unsigned char mg_smem[];
  uint16_t* row = (uint16_t*)mg_smem;
  const int t = threadIdx.x;
  const int total = min(*ntpp, n_sorted);
  const int pieces = size_k >> 3;
  for (int slot = blockIdx.x; slot < total; slot += gridDim.x) {
    const int id = sorted_ids[slot];
    const int e = expert_ids[slot / block];
    if ((unsigned)id >= (unsigned)c_rows || e < 0) continue;  // (uniform over the workgroup)
    const uint16_t* src = a + (int64_t)(id / top_k) * lda;
    const int32_t* pe = perm + (int64_t)e * size_k;
    uint16_t* dst = out + (int64_t)slot * size_k;
    if constexpr (STAGED) {
      __syncthreads();  // the previous turn's gathers are done
      for (int p = t; p < pieces; p += 256) ((u32x4*)row)[p] = ((const u32x4*)src)[p];
      __syncthreads();
      for (int p = t; p < pieces; p += 256) {
        const u32x4 i0 = *(const u32x4*)(pe + 8 * p), i1 = *(const u32x4*)(pe + 8 * p + 4);
        u32x4 v;
        v[0] = (uint32_t)row[i0[0]] | ((uint32_t)row[i0[1]] << 16);
        v[1] = (uint32_t)row[i0[2]] | ((uint32_t)row[i0[3]] << 16);
        v[2] = (uint32_t)row[i1[0]] | ((uint32_t)row[i1[1]] << 16);
        v[3] = (uint32_t)row[i1[2]] | ((uint32_t)row[i1[3]] << 16);
        ((u32x4*)dst)[p] = v;
      }
    } else {
      for (int k = t; k < size_k; k += 256) dst[k] = src[pe[k]];
    }
  }
}

int moe_gather_rows(const w4a16_gemm_args* a, void* out, hipStream_t stream) {
  const int64_t k = a->size_k;
  if (a->n_sorted <= 0 || k == 0) return 0;
  const int64_t slots = a->n_sorted;
  const unsigned grid = (unsigned)(slots < 8 * (int64_t)num_cus() ? slots : 8 * (int64_t)num_cus());
  const int c_rows = (int)(a->size_m * a->top_k);
  const bool staged = k % 8 == 0 && k <= MG_MAX_K && a->lda % 8 == 0 && ((uintptr_t)a->a & 15) == 0 &&
                      ((uintptr_t)out & 15) == 0 && ((uintptr_t)a->perm & 15) == 0;
  if (staged)
    moe_gather_rows_kernel<true><<<grid, 256, (size_t)k * 2, stream>>>(
        (const uint16_t*)a->a, a->lda, a->perm, a->sorted_token_ids, a->expert_ids, a->num_tokens_past_padded,
        (int)a->n_sorted, a->moe_block_size, a->top_k, c_rows, (int)k, (uint16_t*)out);
  else
    moe_gather_rows_kernel<false><<<grid, 256, 0, stream>>>(
        (const uint16_t*)a->a, a->lda, a->perm, a->sorted_token_ids, a->expert_ids, a->num_tokens_past_padded,
        (int)a->n_sorted, a->moe_block_size, a->top_k, c_rows, (int)k, (uint16_t*)out);
  W4A16_HIP(hipGetLastError());
  return 0;
}
}  // namespace w4a16

extern "C" int w4a16_moe_sum(const void* in, void* out, int64_t tokens, int32_t top_k, int64_t hidden,
                             int32_t dtype, void* stream) {
  W4A16_CHECK(in && out, "null pointer");
  W4A16_CHECK(hidden % 8 == 0, "hidden = %lld must be divisible by 8", (long long)hidden);
  W4A16_CHECK(dtype == W4A16_DTYPE_F16 || dtype == W4A16_DTYPE_BF16, "unsupported dtype");
  const int64_t total8 = tokens * (hidden / 8);
  if (total8 == 0) return 0;
  const int64_t blocks = ceil_div(total8, 256);
  const unsigned grid = (unsigned)(blocks < 65536 ? blocks : 65536);
  if (dtype == W4A16_DTYPE_F16)
    moe_sum_kernel<DT_F16><<<grid, 256, 0, (hipStream_t)stream>>>((const uint16_t*)in, (uint16_t*)out, total8, top_k, hidden / 8);
  else
    moe_sum_kernel<DT_BF16><<<grid, 256, 0, (hipStream_t)stream>>>((const uint16_t*)in, (uint16_t*)out, total8, top_k, hidden / 8);
  W4A16_HIP(hipGetLastError());
  return 0;
}

extern "C" int w4a16_silu_and_mul(const void* in, void* out, int64_t tokens, int64_t d, int32_t dtype,
                                  void* stream) {
  W4A16_CHECK(in && out, "null pointer");
  W4A16_CHECK(d % 8 == 0, "d = %lld must be divisible by 8", (long long)d);
  W4A16_CHECK(dtype == W4A16_DTYPE_F16 || dtype == W4A16_DTYPE_BF16, "unsupported dtype");
  const int64_t total8 = tokens * (d / 8);
  if (total8 == 0) return 0;
  const int64_t blocks = ceil_div(total8, 256);
  const unsigned grid = (unsigned)(blocks < 65536 ? blocks : 65536);
  if (dtype == W4A16_DTYPE_F16)
    silu_and_mul_kernel<DT_F16><<<grid, 256, 0, (hipStream_t)stream>>>((const uint16_t*)in, (uint16_t*)out, total8, d / 8);
  else
    silu_and_mul_kernel<DT_BF16><<<grid, 256, 0, (hipStream_t)stream>>>((const uint16_t*)in, (uint16_t*)out, total8, d / 8);
  W4A16_HIP(hipGetLastError());
  return 0;
}

extern "C" int w4a16_topk_softmax(const void* gating_output, int32_t gating_dtype, float* topk_weights,
                                  int32_t* topk_ids, int32_t* token_expert_indices, int64_t num_tokens,
                                  int32_t num_experts, int32_t topk, int32_t renormalize, void* stream) {
  W4A16_CHECK(gating_output && topk_weights && topk_ids && token_expert_indices, "null pointer");
  W4A16_CHECK(num_experts >= 1 && num_experts <= 64 * TOPK_PER_LANE, "num_experts = %d must be in [1, %d]", num_experts,
              64 * TOPK_PER_LANE);
  W4A16_CHECK(topk >= 1 && topk <= num_experts, "topk = %d must be in [1, num_experts]", topk);
  W4A16_CHECK(num_tokens >= 0 && num_tokens < (1LL << 30), "bad num_tokens");
  if (num_tokens == 0) return 0;
  hipStream_t st = (hipStream_t)stream;
  if (gating_dtype == W4A16_DTYPE_F16)
    launch_topk<_Float16>(gating_output, topk_weights, topk_ids, token_expert_indices, num_tokens, num_experts, topk, renormalize, st);
  else if (gating_dtype == W4A16_DTYPE_BF16)
    launch_topk<__bf16>(gating_output, topk_weights, topk_ids, token_expert_indices, num_tokens, num_experts, topk, renormalize, st);
  else if (gating_dtype == W4A16_DTYPE_F32)
    launch_topk<float>(gating_output, topk_weights, topk_ids, token_expert_indices, num_tokens, num_experts, topk, renormalize, st);
  else
    return fail(W4A16_EINVAL, "gating_output must be fp16, bf16 or fp32");
  W4A16_HIP(hipGetLastError());
  return 0;
}

extern "C" int w4a16_batched_moe_align_block_size(int64_t max_tokens_per_batch, int32_t block_size,
                                                  const int32_t* batch_num_tokens, int32_t num_batches,
                                                  int32_t* sorted_ids, int64_t sorted_len, int32_t* block_ids,
                                                  int64_t block_ids_len, int32_t* num_tokens_post_pad, void* stream) {
  W4A16_CHECK(batch_num_tokens && sorted_ids && block_ids && num_tokens_post_pad, "null pointer");
  W4A16_CHECK(block_size > 0 && max_tokens_per_batch >= 0, "bad block_size / max_tokens_per_batch");
  W4A16_CHECK(num_batches >= 1 && num_batches <= ALIGN_MAX_EXPERTS, "num_batches = %d must be in [1, %d]", num_batches,
              ALIGN_MAX_EXPERTS);
  const int64_t want = ceil_div(max_tokens_per_batch, block_size) * block_size * num_batches;
  W4A16_CHECK(sorted_len == want, "sorted_ids has %lld elements, expected %lld", (long long)sorted_len, (long long)want);
  W4A16_CHECK(block_ids_len == want / block_size, "batch_ids has %lld elements, expected %lld", (long long)block_ids_len,
              (long long)(want / block_size));
  W4A16_CHECK(want < (1LL << 31) && num_batches * max_tokens_per_batch < (1LL << 31), "problem too large");
  batched_moe_align_kernel<<<1, ALIGN_THREADS, 0, (hipStream_t)stream>>>(num_batches, (int)max_tokens_per_batch, block_size,
                                                                         batch_num_tokens, sorted_ids, (int)sorted_len,
                                                                         block_ids, num_tokens_post_pad);
  W4A16_HIP(hipGetLastError());
  return 0;
}
