// W4A16 GEMM for gfx950 on the 8-bit matrix unit: C[M,N] = A[M,K] * dequant(Bq)[K,N] (+bias), bf16 activations, integer 4-bit
// weights, scale groups of whole 128 K rows (or one scale per column), more than 128 rows.
//
// The 16-bit kernels spend their time on making weights: 4.25 VALU instructions per pair of bf16((q - z) * s), which a SIMD barely
// overlaps with its MFMAs (prefill kernel, 4096^3: matrix pipe 52 % busy).  The 8-bit unit does twice the products per cycle and
// takes the integer q - z as it is, an e4m3 number: 11 instructions make eight of them from a word of uint4b8 codes, 16 with zero points
// (x8_weights).  The activation becomes two e4m3 terms under one power of two per row and 128 K rows ("step"): hi = e4m3(a * 2^-e),
// lo = e4m3(32 * (a * 2^-e - hi)).  bf16 has eight significant bits, the terms four each: the pair is the activation, exactly, down to
// 2^-15 of the step's largest value, and has an absolute error of 2^-23 of that below.  Two v_mfma_scale_f32_16x16x128_f8f6f4 (hi, lo;
// same weights) do what four bf16 MFMAs did, in the same 64 cycles; the step's sums are then scaled in fp32, acc = fma(s, sum, acc), so no
// weight is rounded.  Where an outlier leaves eight neighbours of its row and step more than 13 binades below it, what the terms leave out
// of that row is added by the 16-bit unit behind the loop ("wide" steps): otherwise a term's error is below 2^-9 of the largest of eight
// neighbours, no more than rounding their weights to bf16 costs.  A column whose weights at the large values are zero sees the small ones alone, so
// a step is also wide where a value loses bits and fewer than 32 of the 128 are within 13 binades of the largest (sparse rows; 2^13 with 1 and 2^-12
// side by side: the 2^-12 was lost).  With 32 and more, only a column whose weights are zero at all of them shows the loss: 2^-23 of the
// largest value.  (Normal activations have 120 and more there, and the test costs the split pass 2 %; with a quarter of 4096 x 4096 activations not
// zero, 32 to a step, the sums behind the loop go from 200 to 380 us beside 730, with a tenth from 200 to 290.)  4096 x 28672 at 203 rows, 59 us: one
// wide step of one row 64, one feature 1000 times the others 59, 10^5 times 73 (one wide step in every row), eight of them 152, one in every step
// 430.
//   Measured on the unit: subnormals are kept; lane l holds row / column l & 15 and the 32 bytes of K block l >> 4, one scale byte
// per row serves the whole step when all four lanes of the row carry it; products of eight neighbouring bytes are added with the bits
// below 2^-14 of the largest cut off, these sums then in fp32.  What counts as large is the sum of the two exponents, a subnormal's being
// that of the smallest normal number; a zero factor does not count.  Hence the weights' form: signed, with their zero point taken off, so
// that a weight of value zero adds exactly zero whatever it meets, and not far below the normal numbers (uint4b8: 2 (q - 8), 4 .. 8 are
// normal; zero points: all of them).  Error of a column against float64, K = 4096, normal activations but for one feature 1000 times the
// others: 1.66e-3 where its weight there is zero, 1.70e-3 where that is +-1 (uint4b8; 1.66e-3 zero points), 1.66e-3 elsewhere and without
// the outlier (rounding the result to bf16 alone: 1.66e-3; 16-bit kernels: 2.13e-3, 1.67e-3, and up to 2.4e-3 by the weight's rounding).
// What this form avoids: unsigned codes with -z * (sum of a) added back, 7.0e-3 where the weight is zero (5.5e-2 with an outlier of 10000);
// q - 8 in units of the smallest subnormal, 1.86e-3 where it is +-1.  It costs 1 % (uint4b8) and 4 % (zero points) of a long launch.
//
//   split    x8_split_kernel writes the two terms of A in the order in which MFMA fragments are read (a fragment of 16 rows is one
//            contiguous KB) with the scale bytes of every row and step: 16 us at 4096 x 4096, 44 at 4096 x 14336 (5 TB/s).
//   tile     a wavefront owns 16 MB rows x 64 columns (half of the words of a column pair): 128 accumulators at MB = 8, two
//            wavefronts per SIMD, every register used.  The accumulators must be VGPRs (the VALU cannot add to AGPRs).
//   shapes   <8, KS 1, WN 8>: 128 x 512, one workgroup per compute unit; <8, 1, 4>: 128 x 256, two; <5 .. 8, 2, 4>: 80 .. 128 rows x 256
//            columns, K in two halves inside the workgroup, for problems that leave compute units idle otherwise.  gemm.hip picks by
//            a fitted cost.
//   staging  activations global -> LDS without registers, double buffered, one barrier per step, placed where a wavefront has read
//            the last fragment of its step.  Addresses decide the rate: one KB costs the compute unit's memory pipe 17 cycles read
//            contiguously, 64 in rows of 64 bytes (the first layout tried: 128 x 256 tiles with K halves 937 us, 815 with this one).
//            Weights global -> registers, one step ahead, spread over the step (a wavefront whose load finds the queue full stands
//            still).  Through LDS they cost more there than they save in the memory pipe (128 rows: 108 -> 114 us).
//   prepared Zero points make a weight 16 instructions of eight, which a long launch pays once per 128 rows of A: x8_weights_kernel writes the e4m3
//            numbers once, in operand order (4096 x 28672: 40 us, 176 MB moved at 4.4 TB/s), and x8_prepared_kernel loads them; 2.3 other VALU
//            instructions per MFMA are left, the folds.  4096 x 28672 at 4096 rows 786 -> 694 us, 14336 x 4096 at 3000 rows 350 -> 307; the GEMM
//            alone is at 1.51 to 1.59 PFLOP/s, near what the power limit leaves of the MFMAs (1.65).  uint4b8 gains 3 % at most and stays.
//   bound    4096 x 28672 bf16, weights not cached, 16-bit kernels and this one: at 4096 rows uint4b8 799 -> 731 us, zero points 812 -> 811; at
//            1024 rows 225 -> 201 and 226 -> 222; at 203 rows 68.5 -> 58.6 and 67.9 -> 61.8.  Long launches: matrix pipe 54 % (48 % with zero
//            points) of the cycles at 2.1 GHz, 5.3 (6.8) other VALU instructions per MFMA of twice a 16-bit one's time, a third of which it
//            overlaps; the MFMAs with their FMAs alone are held to 1.54 GHz by the power limit, 1.65 PFLOP/s.  One-round launches: MFMA,
//            start and end of the workgroups, the split pass.
#include <type_traits>

#include "gemm_kernels.h"

namespace w4a16 {

using i32x8 = int32_t __attribute__((ext_vector_type(8)));
using u16x2 = uint16_t __attribute__((ext_vector_type(2)));

constexpr int X8_G = 128;                       // K rows of one step
constexpr int X8_RS = 76;                       // floats per row of an epilogue slab (40 per n-tile half: conflict-free, 16-byte aligned)
constexpr int X8_SLAB = 2 * 16 * X8_RS * 4;     // a wavefront's two slabs of 16 rows

__host__ __device__ constexpr int x8_buf(int mb, int wn) { return mb * 4096 + wn * 256; }  // one K part, one step: fragments, scales
__host__ __device__ constexpr int x8_smem(int mb, int ks, int wn) {
  const int bufs = 2 * ks * x8_buf(mb, wn), comb = (ks - 1) * ks * wn * ((mb + ks - 1) / ks) * 4096, slabs = ks * wn * X8_SLAB;
  return bufs > comb ? (bufs > slabs ? bufs : slabs) : (comb > slabs ? comb : slabs);
}
constexpr int X8_TABLES = 16 * 16;  // behind it, with zero points: a table for each

constexpr int X8_WIDE = 13;         // binades from a step's largest value at which what the two terms leave out is added
constexpr int X8_EXACT = 14;        // binades from it down to which the two terms leave nothing out
constexpr int X8_FEW = 32;          // and it is added, too, where fewer values than this are within X8_WIDE

// prepared weights of one step: 8 KB for each unit, two units for every column pair (whose second n-tile may be missing)
__host__ __device__ constexpr int64_t x8_weight_step(int64_t n) { return (n + 127) / 128 * 16384; }

struct X8Params {
  KParams k;
  const unsigned char* w8;   // prepared weights (x8_weights_kernel), or null
  const unsigned char* rec;  // [K / 128][rows / 16][fragment 4][K group 4][row 16][16 bytes]: a fragment is one contiguous KB
  const uint32_t* scl;       // [K / 128][rows]
  int rows;                  // see x8_rows
};
// rows the split activations have: whole blocks of 16, and seven blocks more (a tile starts inside the matrix, and has up to eight)
__host__ __device__ constexpr int64_t x8_rows(int64_t m) { return (m + 15) / 16 * 16 + 112; }

// ------------------------------------------------------------------------------------------------ activations
// A workgroup: 16 rows, wavefront w rows 4 w .. 4 w + 3, X8_SG steps one after the other (their loads are issued together).
// Lane bits: 0 odd half of a k-tile, 1 which four k-tiles, 2-3 row, 4-5 k-tile.
// MoE: row r is that of slot r, read through sorted_ids (slots without a token: zeros), or the slot's own where the rows were gathered; rows behind
// the last live block of 128 are never read, and not written.
struct X8Slots {
  const int32_t *ids, *ntpp;
  int n_sorted, c_rows, top_k, by_slot;
};
template <int X8_SG, bool MOE>
__device__ __forceinline__ void x8_split(const uint16_t* a, int64_t lda, int rows, int stride, int groups, unsigned char* rec, uint32_t* scl,
                                         const X8Slots& slots) {
  if (MOE && (int)blockIdx.x * 16 >= (*slots.ntpp + 127) / 128 * 128) return;
  const int lane = threadIdx.x & 63;
  const int odd = lane & 1, j = (lane >> 1) & 1, rr = lane >> 4;
  const int row = blockIdx.x * 16 + (threadIdx.x >> 6) * 4 + ((lane >> 2) & 3);
  const int group0 = blockIdx.y * X8_SG;
  int64_t src = row < rows ? row : -1;
  if constexpr (MOE) {
    const int id = row < slots.n_sorted ? slots.ids[row] : -1;
    src = (unsigned)id >= (unsigned)slots.c_rows ? -1 : slots.by_slot ? row : id / slots.top_k;
  }
  __shared__ __align__(16) unsigned char sh[X8_SG * 4096];
  u32x4 xs[X8_SG];
#pragma unroll
  for (int q = 0; q < X8_SG; ++q) {
    xs[q] = u32x4{0, 0, 0, 0};
    if (group0 + q < groups && src >= 0) xs[q] = *(const u32x4*)(a + src * lda + (group0 + q) * X8_G + (4 * j + rr) * 16 + odd * 8);
  }
#pragma unroll
  for (int q = 0; q < X8_SG; ++q) {
    const int group = group0 + q;
    if (group >= groups) break;  // (uniform)
    u32x4 x = xs[q];
    // maximum (as 15-bit integers: the order of the magnitudes) over the step's 16 lanes: bits 0, 1, 4, 5
    uint32_t mine = 0;  // (of the lane's own eight)
    auto max_abs = [&](const u32x4& v) {
      u16x2 t = __builtin_bit_cast(u16x2, v[0] & 0x7fff7fffu);
#pragma unroll
      for (int i = 1; i < 4; ++i) t = __builtin_elementwise_max(t, __builtin_bit_cast(u16x2, v[i] & 0x7fff7fffu));
      mine = max((uint32_t)t.x, (uint32_t)t.y);
      uint32_t m = max(mine, (uint32_t)__builtin_amdgcn_mov_dpp((int)mine, 0xb1, 0xf, 0xf, true));
      m = max(m, (uint32_t)__builtin_amdgcn_mov_dpp((int)m, 0x4e, 0xf, 0xf, true));
      const auto p = __builtin_amdgcn_permlane16_swap(m, m, false, false);
      m = max(p[0], p[1]);
      const auto r = __builtin_amdgcn_permlane32_swap(m, m, false, false);
      return max(r[0], r[1]);
    };
    uint32_t m = max_abs(x), flags = 0;
    if (__any(m >= 0x7f80u)) {
      // a NaN stays one in both terms and makes its row's results NaN; infinities, which e4m3 does not have, leave the operand, and the
      // GEMM's epilogue puts them back (x8_infinite_row)
      u32x4 finite = x;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t lo = x[i] & 0x7fffu, hi = (x[i] >> 16) & 0x7fffu;
        if (lo >= 0x7f80u) flags |= lo == 0x7f80u ? 1u : 2u, finite[i] &= 0xffff0000u;
        if (hi >= 0x7f80u) flags |= hi == 0x7f80u ? 1u : 2u, finite[i] &= 0x0000ffffu;
        if (lo == 0x7f80u) x[i] &= 0xffff0000u;
        if (hi == 0x7f80u) x[i] &= 0x0000ffffu;
      }
      flags |= (uint32_t)__shfl_xor((int)flags, 1);
      flags |= (uint32_t)__shfl_xor((int)flags, 2);
      flags |= (uint32_t)__shfl_xor((int)flags, 16);
      flags |= (uint32_t)__shfl_xor((int)flags, 32);
      m = max_abs(finite);
    }
    // wide step: eight neighbours below 2^-X8_WIDE of the row's largest value (not zeros: those are exact), see x8_rest
    const bool wide = mine != 0 && (int)mine < (int)m - (X8_WIDE << 7);
    const uint64_t row_lanes = 0x000f000f000f000full << (lane & 12);
    if (__ballot(wide) & row_lanes) flags |= 4u;
    // ... or a value that loses bits in a step with few large ones: a column whose weights at those are zero has nothing else to show
    u16x2 least = {0xffff, 0xffff};  // of the lane's magnitudes that are not zero, less one
#pragma unroll
    for (int i = 0; i < 4; ++i) least = __builtin_elementwise_min(least, __builtin_bit_cast(u16x2, x[i] & 0x7fff7fffu) - u16x2{1, 1});
    const uint64_t lossy = __ballot((int)min((uint32_t)least.x, (uint32_t)least.y) + 1 < ((int)(m >> 7) - X8_EXACT) << 7);
    if (lossy) {
      int large = 0;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int mag = (int)(x[i >> 1] >> (16 * (i & 1)) & 0x7fffu);
        large += __popcll(__ballot(mag >= (int)m - (X8_WIDE << 7)) & row_lanes);
      }
      if (large < X8_FEW && (lossy & row_lanes)) flags |= 4u;
    }
    const int e = max((int)(m >> 7) - 134, -122);  // |a| * 2^-e < 256
    const float inv = __builtin_bit_cast(float, (uint32_t)(127 - e) << 23);
    uint32_t hi01 = 0, hi23 = 0, lo01 = 0, lo23 = 0;
    // element pair g of the lane: K rows 2g, 2g + 1 (+ 8 for odd lanes) of its k-tile; two bytes per pair
    auto enc = [&](uint32_t pair, uint32_t& h, uint32_t& l, auto upper_tag) {
      constexpr bool UPPER = decltype(upper_tag)::value;
      const float x0 = bf16_lo_f32(pair), x1 = bf16_hi_f32(pair);
      const float y0 = x0 * inv, y1 = x1 * inv;
      h = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(y0, y1, (int)h, UPPER);
      const auto b = __builtin_amdgcn_cvt_pk_f32_fp8((int)h, UPPER);
      l = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32((y0 - b[0]) * 32.f, (y1 - b[1]) * 32.f, (int)l, UPPER);
    };
    enc(x[0], hi01, lo01, std::false_type{});
    enc(x[1], hi01, lo01, std::true_type{});
    enc(x[2], hi23, lo23, std::false_type{});
    enc(x[3], hi23, lo23, std::true_type{});
    // even lanes collect pairs 0, 1 of both halves, odd lanes pairs 2, 3: bytes [k, k + 1, k + 8, k + 9]
    auto join = [&](uint32_t p01, uint32_t p23, uint32_t& d0, uint32_t& d1) {
      const uint32_t got = (uint32_t)__builtin_amdgcn_mov_dpp((int)(odd ? p01 : p23), 0xb1, 0xf, 0xf, true);
      const uint32_t first = odd ? got : p01, second = odd ? p23 : got;
      d0 = __builtin_amdgcn_perm(second, first, 0x05040100u);
      d1 = __builtin_amdgcn_perm(second, first, 0x07060302u);
    };
    uint32_t d[4];
    join(hi01, hi23, d[0], d[1]);
    join(lo01, lo23, d[2], d[3]);
    // transpose over lane bits 4-5: lane rr gets dword rr of the four k-tiles
    auto swap32 = [](uint32_t& p, uint32_t& q) {
      const auto r = __builtin_amdgcn_permlane32_swap(p, q, false, false);
      p = r[0], q = r[1];
    };
    auto swap16 = [](uint32_t& p, uint32_t& q) {
      const auto r = __builtin_amdgcn_permlane16_swap(p, q, false, false);
      p = r[0], q = r[1];
    };
    swap32(d[0], d[2]);
    swap32(d[1], d[3]);
    swap16(d[0], d[1]);
    swap16(d[2], d[3]);
    // (fragment, K group, row) of the lane's 16 bytes; stored below, a fragment per wavefront
    *(u32x4*)(sh + q * 4096 + ((rr >> 1) * 2 + j) * 1024 + (2 * odd + (rr & 1)) * 256 + (row & 15) * 16) = u32x4{d[0], d[1], d[2], d[3]};
    if ((lane & 0x33) == 0) scl[(int64_t)group * stride + row] = (uint32_t)(127 + e) | (uint32_t)(127 + e - 5) << 8 | flags << 16;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < X8_SG; ++q)
    if (group0 + q < groups)
      *(u32x4*)(rec + ((int64_t)(group0 + q) * stride + blockIdx.x * 16) * 256 + threadIdx.x * 16) = *(const u32x4*)(sh + q * 4096 + threadIdx.x * 16);
}

template <int X8_SG>
__global__ __launch_bounds__(256) void x8_split_kernel(const uint16_t* a, int64_t lda, int rows, int stride, int groups, unsigned char* rec,
                                                       uint32_t* scl) {
  asm volatile("" ::"s"(a), "s"(lda), "s"(rows), "s"(stride), "s"(groups), "s"(rec), "s"(scl));  // (the arguments in one turn, not three)
  x8_split<X8_SG, false>(a, lda, rows, stride, groups, rec, scl, X8Slots{});
}
__global__ __launch_bounds__(256) void x8_split_slots_kernel(const uint16_t* a, int64_t lda, int stride, int groups, unsigned char* rec, uint32_t* scl,
                                                             const X8Slots slots) {
  x8_split<4, true>(a, lda, 0, stride, groups, rec, scl, slots);
}

// ------------------------------------------------------------------------------------------------ GEMM
// What the infinities (and NaNs) of one row of A in steps [g0, g1) add up to in columns n .. n + 3 of each of 16 lanes: the row's results,
// whatever else it holds.  `flags`: the row's scale words, a stride of `rows` apart.  The 16 lanes look through the flags of 16 steps
// together and through a flagged step's 128 elements together, until all their sums are NaN.
template <bool ZP, bool CHANNEL>
__device__ __forceinline__ f32x4 x8_infinite_row(const uint16_t* arow, const uint32_t* flags, int rows, int g0, int g1, const uint32_t* Bq,
                                                 const uint16_t* Sc, const uint32_t* Zp, int N, int group_shift, int n) {
  const int lane = threadIdx.x & 63, l16 = lane & 15;
  auto mine = [&](bool b) { return (uint32_t)(__ballot(b) >> (lane & 48)) & 0xffffu; };  // a bit for each of the 16 lanes
  f32x4 v = {0, 0, 0, 0};
  auto all_nan = [&]() { return v[0] != v[0] && v[1] != v[1] && v[2] != v[2] && v[3] != v[3]; };
  auto add = [&](int k) {
    const float av = __builtin_bit_cast(float, (uint32_t)arow[k] << 16);
    const int grp = CHANNEL ? 0 : (k >> 5) >> group_shift;
    const int r = k & 15, g = (r & 7) >> 1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int col = n + i, cc = col & 63, w = cc >> 4, half = (cc >> 3) & 1, c = cc & 7;
      const uint32_t word = Bq[(int64_t)(k >> 4) * (2 * N) + (col >> 6) * 128 + (4 * c + g) * 4 + w];
      const int q = (int)((word >> (4 * ((r & 1) * 4 + half * 2 + (r >> 3)))) & 15u);
      int z = 8;
      if (ZP) z = (int)((Zp[(int64_t)grp * (N >> 3) + (col >> 6) * 8 + c] >> (4 * w + 16 * half)) & 15u);
      float s = 1.f;
      if (!CHANNEL) s = bf16_lo_f32(Sc[(int64_t)grp * N + (col & ~63) + 8 * c + 2 * w + half]);
      v[i] += av * ((float)(q - z) * s);
    }
  };
#pragma unroll 1
  for (int gi = g0; gi < g1 && mine(!all_nan()); gi += 16) {
    uint32_t steps = mine(gi + l16 < g1 && (flags[(int64_t)min(gi + l16, g1 - 1) * rows] >> 16 & 3u) != 0);
#pragma unroll 1
    for (; steps && mine(!all_nan()); steps &= steps - 1) {
      const int k0 = (gi + __builtin_ctz(steps)) * X8_G;
      const u32x4 x = *(const u32x4*)(arow + k0 + 8 * l16);
#pragma unroll 1
      for (int e = 0; e < 8; ++e) {
        const uint32_t pair = e < 4 ? (e < 2 ? x[0] : x[1]) : (e < 6 ? x[2] : x[3]);
        uint32_t hits = mine(((e & 1 ? pair >> 16 : pair) & 0x7fffu) >= 0x7f80u);
#pragma unroll 1
        for (; hits && !all_nan(); hits &= hits - 1) add(k0 + 8 * __builtin_ctz(hits) + e);
      }
    }
  }
  return v;
}

// What the two terms of bf16 elements (low and high half of `pair`) leave out, as bf16, exactly: a multiple of the element's last bit that
// is smaller than the element.  exp: low byte of the row's scale word.  (The split kernel's encoding; infinities and NaNs leave nothing.)
__device__ __forceinline__ uint32_t x8_rest(uint32_t pair, uint32_t exp) {
  const float inv = __builtin_bit_cast(float, (254u - exp) << 23), x[2] = {bf16_lo_f32(pair), bf16_hi_f32(pair)};
  const float y0 = x[0] * inv, y1 = x[1] * inv;
  const int h = __builtin_amdgcn_cvt_pk_fp8_f32(y0, y1, 0, false);
  const auto hf = __builtin_amdgcn_cvt_pk_f32_fp8(h, false);
  const float d[2] = {y0 - hf[0], y1 - hf[1]};
  const int l = __builtin_amdgcn_cvt_pk_fp8_f32(d[0] * 32.f, d[1] * 32.f, 0, false);
  const auto lf = __builtin_amdgcn_cvt_pk_f32_fp8(l, false);
  const float r[2] = {d[0] - lf[0] * 0x1.0p-5f, d[1] - lf[1] * 0x1.0p-5f}, back = __builtin_bit_cast(float, exp << 23);
  float out[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    // (an element too small for either term is left out whole, and y may have lost bits of it)
    const bool none = (((h | l) >> (8 * i)) & 0x7f) == 0;
    out[i] = ((pair >> (16 * i)) & 0x7fffu) >= 0x7f80u ? 0.f : none ? x[i] : r[i] * back;
  }
  return pack_bf16(out[0], out[1]);
}

// One 16- or 4-byte piece per lane, global memory -> LDS (lane l's piece at lds + 16 l or 4 l) without passing through registers.
// The statements are opaque to the compiler: whoever reads the data waits for vmcnt(0) and then at a workgroup barrier.
__device__ __forceinline__ void x8_load_lds16(uint32_t lds, uint32_t off, const void* base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ void x8_load_lds4(uint32_t lds, uint32_t off, const void* base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory", "m0");
}

// A word of eight weights -> two operand dwords, of the column in nibbles 0, 1, 4, 5 and of the one in nibbles 2, 3, 6, 7.
// uint4b8: 2 (q - 8) * 2^-9.  (bitop3 by hand: the compiler makes two instructions of either)
__device__ __forceinline__ void x8_weights(uint32_t x, int& o0, int& o1) {
  auto select = [](uint32_t mask, uint32_t a, uint32_t b) { return (uint32_t)__builtin_amdgcn_bitop3_b32(mask, a, b, 0xca); };
  // nibbles: negative where bit 3 is clear (neg: 8 there); magnitude q ^ 8, or (q ^ 7) + 1
  const uint32_t neg = __builtin_amdgcn_bitop3_b32(0x88888888u, x, x, 0x30), one = neg >> 3;  // 0x88888888 & ~x
  const uint32_t mag = (x ^ (0x88888888u - one)) + one;
  const uint32_t lo = select(0x1e1e1e1eu, mag << 1, neg << 4), hi = select(0x1e1e1e1eu, mag >> 3, neg);
  o0 = (int)__builtin_amdgcn_perm(hi, lo, 0x06040200u);
  o1 = (int)__builtin_amdgcn_perm(hi, lo, 0x07050301u);
}
// Zero points: (q - z) * 2^-6, read from the columns' tables t0, t1.
__device__ __forceinline__ void x8_weights(uint32_t x, const u32x4& t0, const u32x4& t1, int& o0, int& o1) {
  const uint32_t lo = x & 0x07070707u, hi = (x >> 4) & 0x07070707u;
  const uint32_t s0 = __builtin_amdgcn_perm(hi, lo, 0x06040200u), s1 = __builtin_amdgcn_perm(hi, lo, 0x07050301u);
  // bytes of ones where bit 3 of the code is set (selectors 8 .. 11: bits 15 and 31 of the second and of the first operand, eight times)
  const uint32_t m0 = __builtin_amdgcn_perm(x << 8, x << 12, 0x0b0a0908u), m1 = __builtin_amdgcn_perm(x, x << 4, 0x0b0a0908u);
  auto entry = [](const u32x4& t, uint32_t s, uint32_t m) {  // (m & upper) | (~m & lower)
    return __builtin_amdgcn_bitop3_b32(m, __builtin_amdgcn_perm(t[3], t[2], s), __builtin_amdgcn_perm(t[1], t[0], s), 0xca);
  };
  o0 = (int)entry(t0, s0, m0), o1 = (int)entry(t1, s1, m1);
}
// Dword `dword` of the table of zero point z: the e4m3 numbers (q - z) * 2^-6, q = 4 dword .. 4 dword + 3.
__device__ __forceinline__ uint32_t x8_table(int z, int dword) {
  uint32_t r = 0;
  for (int i = 0; i < 4; ++i) {
    const int v = 4 * dword + i - z, a = v < 0 ? -v : v, e = a >= 8 ? 3 : a >= 4 ? 2 : a >= 2 ? 1 : 0;
    if (a) r |= ((v < 0 ? 0x80u : 0u) | (uint32_t)(e + 1) << 3 | ((uint32_t)a << (3 - e) & 7u)) << (8 * i);
  }
  return r;
}

template <bool ZP, bool CHANNEL, int MB, int KS, int WN, bool PREP, bool MOE = false>
__device__ __forceinline__ void x8_tile(const X8Params& xp) {
  const KParams& p = xp.k;
  constexpr int BM = 16 * MB, BN = WN * 64;
  constexpr int NL = MB * 4 / WN;  // 1 KB fragments staged per wavefront and step
  constexpr int NM = (BM + 63) / 64;          // 64-row pieces of the step's scales
  static_assert(NM <= WN && MB * 4 % WN == 0, "one piece of scales and as many fragments for every wavefront");
  extern __shared__ __align__(16) unsigned char smem[];
  const int t = threadIdx.x, lane = t & 63;
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int part = wv / WN, wn = wv % WN;
  const int c = lane & 7, h = (lane >> 3) & 1, g = lane >> 4;
  const int G = p.K / X8_G;

  int mtiles = (p.M + BM - 1) / BM, nsplit = p.splits;
  int j = blockIdx.x, split = 0, slot = 0;
  int gb = 0, ge = G;
  if constexpr (MOE) {  // (as the prefill kernel: K pieces of the last round's tiles, whole tiles in runs for every XCD)
    static_assert(BM == FB_BM && KS == 1 && BN == 512, "the tiles of the prefill kernel and of its second pass");
    zero_fill_side_job(p);
    mtiles = min((*p.ntpp + BM - 1) / BM, (p.n_sorted + BM - 1) / BM);
    if (mtiles == 0) return;
    const TailSplit d = tail_split(mtiles * p.ncp, p.dyn_slots, p.total_ksteps, FB_MIN_SPLIT);
    nsplit = 1;
    if (j < d.F) {
      if ((d.F & 7) == 0) j = (j & 7) * (d.F >> 3) + (j >> 3);
    } else {
      const int u = j - d.F;
      if (u >= d.R * d.S) return;
      slot = u % d.R, split = u / d.R, nsplit = d.S;
      gb = split * d.kps / 4, ge = min(gb + d.kps / 4, G);
      j = d.F + slot;
    }
  } else if (nsplit > 1) {
    const int tiles = mtiles * p.ncp, per = p.ksteps_per_split / 4;
    split = j / tiles;
    j -= split * tiles;
    slot = j;
    gb = split * per, ge = min(gb + per, G);
  }
  const int gb0 = gb, ge0 = ge;
  const int max_steps = (ge - gb + KS - 1) / KS;  // of a K part
  gb += part * max_steps;
  ge = min(gb + max_steps, ge);
  const int steps = ge - gb;  // the last part may have fewer (or none)
  int mt = j % mtiles, strip = p.strip0 + j / mtiles;
  if (MOE) chunked_tile(j, mtiles, p.ncp, mt, strip);
  const int row0 = mt * BM;
  const int u = strip * WN + wn, cp = u >> 1, wsel = (u & 1) * 2;
  const bool wave_on = cp * 128 < p.N;

  const uint32_t* Bq = p.B;
  const uint16_t* Sc = (const uint16_t*)p.S;
  const uint16_t* bias = (const uint16_t*)p.bias;
  if constexpr (MOE) {
    const int e = p.expert_ids[mt];
    if (e < 0) return;  // expert of another rank
    Bq += e * p.b_estride;
    Sc += e * p.s_estride;
    if (bias) bias += e * p.n_estride;
  }
  const int u_mem = wave_on ? u : 0;
  // (fused SiLU-and-mul: gate n-tile cp paired with the up n-tile of the same output columns, N / 128 + cp)
  const bool act = MOE && p.act;
  const int nt = !wave_on ? 0 : act ? (h ? (p.N >> 7) + cp : cp) : ((2 * cp + h) * 64 < p.N ? 2 * cp + h : 0);
  // byte offsets of the lane; everything else in an address is uniform
  const uint32_t b_off = (uint32_t)(nt * 128 + (4 * c + g) * 4 + wsel) * 4;
  // (nt * 64 + 8 c + 2 wsel) * 2 of the scales; two instructions per step for a register of the loop's 256
  auto s_off = [&]() {
    uint32_t v;
    asm volatile("v_lshrrev_b32 %0, 2, %1" : "=v"(v) : "v"(b_off));
    return (v & ~15u) + 4 * wsel;
  };
  const uint32_t b_row = (uint32_t)p.N * 8;  // bytes of one k-tile
  // buffer resources: 32-bit offsets, nothing per lane but the lane's own (the host checks the sizes)
  const int b_bytes = (int)((uint32_t)(p.K / 16) * b_row), sg = CHANNEL ? 1 : (4 * G) >> p.group_shift;
  const auto b_res = __builtin_amdgcn_make_buffer_rsrc((void*)Bq, 0, b_bytes, 0x00020000);
  const auto s_res = __builtin_amdgcn_make_buffer_rsrc((void*)Sc, 0, sg * p.N * 2, 0x00020000);
  const auto z_res = __builtin_amdgcn_make_buffer_rsrc((void*)p.Z, 0, sg * (p.N / 2), 0x00020000);

  // activations: fragment f = 4 mb + piece, one KB each; f = wn + WN i for this wavefront
  const int64_t a_step = (int64_t)xp.rows * 256;
  const unsigned char* a_ptr = xp.rec + gb * a_step + (int64_t)row0 * 256;
  const uint32_t* m_ptr = xp.scl + (int64_t)gb * xp.rows + row0 + wn % NM * 64;
  unsigned char* pbuf = smem + part * 2 * x8_buf(MB, WN);
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)pbuf);
  // step i of the part -> LDS; complete after sync_stage
  auto stage_frag = [&](int i, int buf, int q) {
    const int f = wn + WN * q;
    x8_load_lds16(lds0 + buf * x8_buf(MB, WN) + f * 1024, lane * 16, a_ptr + i * a_step + f * 1024);
  };
  auto stage_meta = [&](int i, int buf) {  // (wavefronts from NM on: a copy nobody reads)
    uint32_t off;  // (lane * 4, not kept either)
    asm volatile("v_lshrrev_b32 %0, 2, %1" : "=v"(off) : "v"(lane * 16));
    x8_load_lds4(lds0 + buf * x8_buf(MB, WN) + MB * 4096 + wn * 256, off, m_ptr + (int64_t)i * xp.rows);
  };

  // (nt * 8 + c) * 4 of the zero points, likewise
  auto z_off = [&]() {
    uint32_t v;
    asm volatile("v_lshrrev_b32 %0, 4, %1" : "=v"(v) : "v"(b_off));
    return v & ~3u;
  };

  u32x2 raw[8], sraw = {0, 0};
  uint32_t zraw = 0;
  u32x4 tab[2] = {};
  unsigned char* tables = smem + x8_smem(MB, KS, WN);
  if (ZP && !PREP && t < X8_TABLES / 4) ((uint32_t*)tables)[t] = x8_table(t >> 2, t & 3);  // (complete after the first sync_stage)
  auto load_b = [&](int i, int kt) {
    raw[kt] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(b_res, b_off, (uint32_t)((gb + i) * 8 + kt) * b_row, 0));
  };
  auto load_s = [&](int i) {
    const uint32_t grp = CHANNEL ? 0 : (uint32_t)(4 * (gb + i)) >> p.group_shift;
    if (!CHANNEL) sraw = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(s_res, s_off(), grp * p.N * 2, 0));
    if (ZP && !PREP) zraw = __builtin_amdgcn_raw_buffer_load_b32(z_res, z_off(), grp * (p.N / 2), 0);
  };
  // prepared weights: piece q of step i, 16 bytes of operand q >> 1
  const uint64_t w8_step = x8_weight_step(p.N);
  auto load_w8 = [&](int i, int q, i32x8 (&o)[4]) {
    const u32x4 v = *(const u32x4*)(xp.w8 + (uint64_t)(gb + i) * w8_step + (uint64_t)u_mem * 8192 + q * 1024 + lane * 16);
#pragma unroll
    for (int e = 0; e < 4; ++e) o[q >> 1][4 * (q & 1) + e] = (int)v[e];
  };
  // tables of word w's two columns, from the loaded word of zero points
  auto zeros = [&](int w) {
    if (ZP && !PREP) {
      const uint32_t z = zraw >> (4 * (wsel + w));
      tab[0] = *(const u32x4*)(tables + (z & 15u) * 16);
      tab[1] = *(const u32x4*)(tables + (z >> 16 & 15u) * 16);
    }
  };
  // k-tile kt of word w (0 or 1 of the wavefront's two) -> its dword of the two operands
  auto dequant = [&](int w, int kt, auto& o) {
    int o0, o1;
    if constexpr (ZP)
      x8_weights(raw[kt][w], tab[0], tab[1], o0, o1);
    else
      x8_weights(raw[kt][w], o0, o1);
    o[0][kt] = o0, o[1][kt] = o1;
  };

  f32x4 acc[MB][4];
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[m][i] = f32x4{0, 0, 0, 0};
  i32x8 bx[4], by[4], b23[2], ah, al;  // (elements 2 and 3 of the first two: prepared weights, whose b23 is not used)
  f32x4 T[2][2] = {};
  constexpr float UNIT = ZP ? 64.f : 256.f;  // of the weights' e4m3 numbers
  float sc[4] = {UNIT, UNIT, UNIT, UNIT};
  uint32_t any = 0, sl = 0, sl_n = 0;
  auto frag = [&](int buf, int m, int half, i32x8& o) {
    const u32x4* f = (const u32x4*)(pbuf + buf * x8_buf(MB, WN) + m * 4096 + half * 2048) + lane;
    const u32x4 f0 = f[0], f1 = f[64];
#pragma unroll
    for (int q = 0; q < 4; ++q) o[q] = (int)f0[q], o[4 + q] = (int)f1[q];
  };
  auto meta = [&](int buf, int m) {
    const unsigned char* d = pbuf + buf * x8_buf(MB, WN) + MB * 4096;
    sl_n = *(const uint32_t*)(d + (m * 16 + (lane & 15)) * 4);
  };
  // word w's two operands: factors of the step's product sums, from the loaded words
  auto scales = [&](int w) {
    if (!CHANNEL) {
      sc[2 * w] = bf16_lo_f32(sraw[w]) * UNIT;
      sc[2 * w + 1] = bf16_hi_f32(sraw[w]) * UNIT;
    }
  };
  auto fold = [&](int m, int pr, int i) {
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[m][2 * pr + i][r] = __builtin_fmaf(sc[2 * pr + i], T[pr][i][r], acc[m][2 * pr + i][r]);
  };
  auto mfma_lo = [&](int pr, int i, const i32x8& b) {
    T[pr][i] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(al, b, f32x4{0, 0, 0, 0}, 0, 0, 1, (int)sl, 0, 127);
  };
  auto mfma_hi = [&](int pr, int i, const i32x8& b) {
    T[pr][i] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(ah, b, T[pr][i], 0, 0, 0, (int)sl, 0, 127);
  };
  auto sync_stage = [&]() {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

#define X8_SB __builtin_amdgcn_sched_barrier(0)
  auto step = [&](int i, int buf, i32x8 (&b01)[4], i32x8 (&n01)[4]) {
    const i32x8 &b2 = PREP ? b01[2] : b23[0], &b3 = PREP ? b01[3] : b23[1];
    constexpr int FROM = MB > 3 ? MB - 3 : 1, PER = (8 + MB - FROM - 1) / (MB - FROM);  // next step's word 0: spread over the last row blocks
    // The next step's loads, spread over the step: a wavefront whose load finds the memory pipeline's queue full stands still with
    // its MFMAs.  u: 2 m + word; the weight registers are free from u = 1 on and wanted from m = FROM on.
    const int nx = min(i + 1, steps - 1);
    auto loads = [&](int u) {
      constexpr int LAST = PREP ? 2 * MB - 2 : 2 * FROM - 1, WPER = (8 + LAST - 1) / LAST, SPER = (NL + LAST - 1) / LAST;
      if (u == 1) load_s(nx), stage_meta(nx, buf ^ 1);
#pragma unroll
      for (int q = 0; q < WPER; ++q)
        if ((u - 1) * WPER + q < 8) {
          if constexpr (PREP)
            load_w8(nx, (u - 1) * WPER + q, n01);
          else
            load_b(nx, (u - 1) * WPER + q);
        }
#pragma unroll
      for (int q = 0; q < SPER; ++q)
        if ((u - 1) * SPER + q < NL) stage_frag(nx, buf ^ 1, (u - 1) * SPER + q);
    };
    scales(0);
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      // columns of word 0; the product sums of word 1 of the row block before are folded meanwhile
      X8_SB;
      mfma_lo(0, 0, b01[0]);
      fold(m > 0 ? m - 1 : MB - 1, 1, 0);  // (zeros in front of the first step)
      if (m == 0 && !PREP) dequant(1, 0, b23), dequant(1, 1, b23);
      X8_SB;
      mfma_lo(0, 1, b01[1]);
      fold(m > 0 ? m - 1 : MB - 1, 1, 1);
      if (m == 0 && !PREP) dequant(1, 2, b23), dequant(1, 3, b23);
      X8_SB;
      mfma_hi(0, 0, b01[0]);
      if (m == 0) scales(1);
      if (m == 0 && !PREP) dequant(1, 4, b23), dequant(1, 5, b23);
      X8_SB;
      mfma_hi(0, 1, b01[1]);
      if (m + 1 < MB) meta(buf, m + 1);
      if (m == 0 && !PREP) {
        dequant(1, 6, b23), dequant(1, 7, b23);
        X8_SB;
      }
      if (m > 0) loads(2 * m);
#pragma unroll
      for (int q = 0; q < PER; ++q)
        if (!PREP && m >= FROM && (m - FROM) * PER + q < 8) dequant(0, (m - FROM) * PER + q, n01);
      X8_SB;
      // columns of word 1
      loads(2 * m + 1);
      X8_SB;
      if (m == MB - 1) {
        sync_stage();
        meta(buf ^ 1, 0);
        X8_SB;
      }
      mfma_lo(1, 0, b2);
      fold(m, 0, 0);
      X8_SB;
      mfma_lo(1, 1, b3);
      fold(m, 0, 1);
      X8_SB;
      frag(m + 1 < MB ? buf : buf ^ 1, m + 1 < MB ? m + 1 : 0, 1, al);
      mfma_hi(1, 0, b2);
      X8_SB;
      mfma_hi(1, 1, b3);
      any |= sl;
      sl = sl_n;
      X8_SB;
      // tables of the next step's word 0 (zero points loaded since u = 1), and then of its word 1
      if (m == FROM - 1) zeros(0);
      if (m == MB - 1) zeros(1);
      frag(m + 1 < MB ? buf : buf ^ 1, m + 1 < MB ? m + 1 : 0, 0, ah);
    }
  };

  // MoE: C row (-1: none) and routing weight of every row of the tile
  int* s_crow = (int*)(smem + x8_smem(MB, KS, WN));
  float* s_tw = (float*)(s_crow + BM);
  if (MOE && t < BM) {
    const int id = row0 + t < p.n_sorted ? p.sorted_ids[row0 + t] : -1, dst = (unsigned)id < (unsigned)p.c_rows ? id : -1;
    s_crow[t] = dst;
    if (p.mul_topk) s_tw[t] = dst >= 0 ? p.topk_w[dst] : 0.f;
  }

  // ---- prologue and main loop: one step (128 K rows) per barrier
  if (steps > 0) {
#pragma unroll
    for (int q = 0; q < NL; ++q) stage_frag(0, 0, q);
    stage_meta(0, 0);
#pragma unroll
    for (int kt = 0; kt < 8; ++kt) {
      if constexpr (PREP)
        load_w8(0, kt, bx);
      else
        load_b(0, kt);
    }
    load_s(0);
  }
  sync_stage();
  if (steps > 0) {
    zeros(0);
#pragma unroll
    for (int kt = 0; kt < 8; ++kt)
      if (!PREP) dequant(0, kt, bx);
    zeros(1);
    meta(0, 0);
    sl = sl_n;
    frag(0, 0, 1, al);
    frag(0, 0, 0, ah);
  }
#pragma unroll 1
  for (int i = 0; i < max_steps; i += 2) {
    if (i < steps)
      step(i, 0, bx, by);
    else
      sync_stage();
    if (i + 1 >= max_steps) break;
    if (i + 1 < steps)
      step(i + 1, 1, by, bx);
    else
      sync_stage();
  }
  if (steps > 0) {
    fold(MB - 1, 1, 0);
    fold(MB - 1, 1, 1);
  }

  // The arguments used from here on are read again: held over the loop they take scalar registers, and with those spilled a vector register,
  // that it has not got.
  X8Params late;
  {
    auto args = __builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(args));
    __builtin_memcpy(&late, (const void*)args, sizeof(late));
  }

  // the row of A behind row r of the tile (one that has a token)
  auto a_row = [&](int r) {
    int64_t src = row0 + r;
    if (MOE && !late.k.a_by_slot) src = s_crow[r] / late.k.top_k;
    return (const uint16_t*)late.k.A + src * late.k.lda;
  };

  // ---- wide steps: what the two terms of the flagged rows leave out, by the 16-bit unit, behind the loop (activations from A, weights as
  // the integers q - z).  A row's result depends on that row alone, and a wavefront on nothing that others do here.
  auto add_rest = [&](int gi) {
    const uint32_t* flags = late.scl + (int64_t)gi * late.rows + row0;
    uint32_t word[(MB + 1) / 2] = {};  // of two row blocks: the high term's scale, bit 10: wide
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      const uint32_t f = flags[16 * m + (lane & 15)];
      word[m / 2] |= ((f & 0xffu) | (f >> 8 & 0x400u)) << (16 * (m % 2));
    }
#pragma unroll
    for (int kt = 0; kt < 8; ++kt) load_b(gi - gb, kt);
    load_s(gi - gb);
    if (ZP && PREP) zraw = __builtin_amdgcn_raw_buffer_load_b32(z_res, z_off(), (CHANNEL ? 0 : (uint32_t)(4 * gi) >> p.group_shift) * (p.N / 2), 0);
#pragma unroll
    for (int half = 0; half < 2; ++half) {  // (64 K rows at a time, or registers spill)
      u32x4 w[2][4];  // [32 K rows][column]
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int z = ZP ? (int)(zraw >> (4 * (wsel + (i >> 1)) + 16 * (i & 1)) & 15u) : 8;
#pragma unroll
          for (int q = 0; q < 2; ++q) {  // rows 2 g, 2 g + 1 of the k-tile, and eight behind them
            const uint32_t v = raw[4 * half + kt][i >> 1] >> (8 * (i & 1) + 4 * q);
            w[kt >> 1][i][2 * (kt & 1) + q] = pack_bf16((float)((int)(v & 15u) - z), (float)((int)(v >> 16 & 15u) - z));
          }
        }
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        X8_SB;
        const bool mine = (word[m / 2] >> (16 * (m % 2) + 10) & 1u) != 0;  // (rows behind the matrix are zeros, not wide)
        if (!__any(mine)) continue;
        u32x4 a[2] = {};
        if (mine) {
          const uint32_t* src = (const uint32_t*)(a_row(16 * m + (lane & 15)) + gi * X8_G + 64 * half) + g;
#pragma unroll
          for (int q = 0; q < 8; ++q) a[q >> 2][q & 3] = src[4 * q];
#pragma unroll
          for (int q = 0; q < 8; ++q) a[q >> 2][q & 3] = x8_rest(a[q >> 2][q & 3], word[m / 2] >> (16 * (m % 2)) & 0xffu);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const f32x4 v = mfma16x16x32<DT_BF16>(a[1], w[1][i], mfma16x16x32<DT_BF16>(a[0], w[0][i], f32x4{0, 0, 0, 0}));
          const float s = CHANNEL ? 1.f : (i & 1) ? bf16_hi_f32(sraw[i >> 1]) : bf16_lo_f32(sraw[i >> 1]);
#pragma unroll
          for (int q = 0; q < 4; ++q) acc[m][i][q] = __builtin_fmaf(s, v[q], acc[m][i][q]);
        }
      }
    }
  };
  if (__any((any >> 18 & 1u) != 0)) {
#pragma unroll 1
    for (int g0 = gb; g0 < ge; g0 += 8) {
      uint32_t f[8], mask = 0;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const uint32_t* flags = late.scl + (int64_t)min(g0 + q, ge - 1) * late.rows + row0;
        f[q] = flags[lane] | flags[min(64 + lane, BM - 1)];
      }
#pragma unroll
      for (int q = 0; q < 8; ++q)
        if (g0 + q < ge && __any((f[q] >> 18 & 1u) != 0)) mask |= 1u << q;
#pragma unroll 1
      for (; mask; mask &= mask - 1) add_rest(g0 + __builtin_ctz(mask));
    }
  }
  __syncthreads();

  // ---- K parts: every part finishes its share of the row blocks and collects the others' accumulators of it through LDS
  constexpr int MS = (MB + KS - 1) / KS;  // row blocks of a part
  const int m0 = part * MS;
  if constexpr (KS > 1) {
    // piece of row blocks MS * owner .. that part `from` hands over
    auto piece = [&](int owner, int from, int mm, int i) {
      return (f32x4*)smem + (((owner * (KS - 1) + (from - owner - 1 + KS) % KS) * WN + wn) * MS * 4 + mm * 4 + i) * 64 + lane;
    };
    auto hand_over = [&](auto part_tag) {  // (the part as a constant: accumulators are registers)
      constexpr int P = decltype(part_tag)::value;
#pragma unroll
      for (int m = 0; m < MB; ++m)
        if (m / MS != P) {
#pragma unroll
          for (int i = 0; i < 4; ++i) *piece(m / MS, P, m % MS, i) = acc[m][i];
        }
    };
    auto collect = [&](auto part_tag) {
      constexpr int P = decltype(part_tag)::value;
#pragma unroll
      for (int mm = 0; mm < MS; ++mm)
        if (P * MS + mm < MB) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            f32x4 v = acc[P * MS + mm][i];
#pragma unroll
            for (int q = 0; q < KS; ++q)
              if (q != P) v += *piece(P, q, mm, i);
            acc[mm][i] = v;
          }
        }
    };
    static_assert(KS == 2, "two parts");
    // (a wrapper around the two calls would put the accumulators into memory)
    if (part == 0)
      hand_over(std::integral_constant<int, 0>{});
    else
      hand_over(std::integral_constant<int, 1>{});
    any = __syncthreads_or((any >> 16 & 1u) != 0) ? 1u << 16 : 0u;
    if (part == 0)
      collect(std::integral_constant<int, 0>{});
    else
      collect(std::integral_constant<int, 1>{});
    __syncthreads();
  }

  // ---- epilogue: two row blocks at a time, accumulators -> slabs of the wavefront -> rows of 2 x 32 columns, 8-byte stores
  float* slab = (float*)(smem + wv * X8_SLAB);
  const int lc = (lane & 15) * 4, lh = lc >> 5, lpos = lh * 40 + (lc & 31);
  const int ncol = 64 * (2 * cp + lh) + 16 * wsel + (lc & 31);
  const bool col_ok = wave_on && ncol < late.k.N;
  float cs[4] = {1.f, 1.f, 1.f, 1.f}, bs[4] = {0.f, 0.f, 0.f, 0.f};
  auto col_consts = [&](int col, float* sc_out, float* b_out) {
    const int base = col & ~31, cl = col & 31;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (CHANNEL) sc_out[i] = bf16_lo_f32(Sc[base + single_perm_pos(cl + i)]);
      if (bias) b_out[i] = bf16_lo_f32(bias[base + single_perm_pos(cl + i)]);
    }
  };
  // fused SiLU-and-mul (unsplit): lane -> row (lane >> 3) + 8 i, gate columns ac .. ac + 3 of the slab's first 32 and the up columns of the same outputs
  const bool act_now = act && nsplit == 1;
  const int ac = (lane & 7) * 4, ocol = 64 * cp + 16 * wsel + ac;
  float cu[4] = {1.f, 1.f, 1.f, 1.f}, bu[4] = {0.f, 0.f, 0.f, 0.f};
  if (act_now) {
    if (wave_on) {
      col_consts(ocol, cs, bs);
      col_consts((late.k.N >> 1) + ocol, cu, bu);
    }
  } else if (col_ok && !act) {
    col_consts(ncol, cs, bs);
  }
  auto finish_act = [&](int r, f32x4 v, f32x4 w) {
    const int crow = s_crow[r];
    if (crow < 0) return;
    const float tw = late.k.mul_topk ? s_tw[r] : 1.f;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      v[q] = (v[q] * cs[q] + bs[q]) * tw;
      w[q] = (w[q] * cu[q] + bu[q]) * tw;
    }
    store_row4_silu_mul<DT_BF16>(late.k, crow, ocol, v, w);
  };
  auto finish = [&](int r, f32x4 v) {  // r: row of the tile
    if (MOE && s_crow[r] < 0) return;
    if (nsplit > 1) {
      *(f32x4*)(late.k.ctmp + (((int64_t)slot * nsplit + split) * BM + r) * BN + (ncol - strip * BN)) = v;
      return;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = v[q] * cs[q] + bs[q];
    if constexpr (MOE) {
      if (late.k.mul_topk) {
        const float tw = s_tw[r];
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] *= tw;
      }
    }
    store_row4<DT_BF16, MOE>(late.k, MOE ? s_crow[r] : row0 + r, ncol, v);
  };
#pragma unroll
  for (int m = 0; m < MS; m += 2) {
#pragma unroll
    for (int e = 0; e < 2 && m + e < MS; ++e)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) slab[(16 * e + 4 * g + r) * X8_RS + 40 * h + 8 * i + c] = acc[m + e][i][r];
    __builtin_amdgcn_wave_barrier();
    if (MOE && act_now) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float* at = slab + ((lane >> 3) + 8 * i) * X8_RS + ac;
        const f32x4 v = *(const f32x4*)at, w = *(const f32x4*)(at + 40);
        if (wave_on) finish_act(16 * m + (lane >> 3) + 8 * i, v, w);
      }
      __builtin_amdgcn_wave_barrier();
      continue;
    }
    f32x4 v[2 * 4];
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (i < 4 || m + 1 < MS) v[i] = *(const f32x4*)(slab + ((lane >> 4) + 4 * i) * X8_RS + lpos);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = (m0 + m) * 16 + (lane >> 4) + 4 * i;
      if ((i < 4 || m + 1 < MS) && r < BM && col_ok && (MOE || row0 + r < late.k.M)) finish(r, v[i]);
    }
    __builtin_amdgcn_wave_barrier();
  }
  if (wave_on && __any((any >> 16 & 1u) != 0)) {
    // rows with infinities, four at a time: 16 lanes have those of theirs that the same lanes have stored above
    const uint32_t* flags = late.scl + row0;
    const int rows = MOE ? BM : min(min(BM, (m0 + MS) * 16), late.k.M - row0);  // of the tile, in front of the part's end
    const int n_in = 128 * cp + 16 * wsel + (lc & 31);          // (lanes whose columns are behind the matrix look along)
    // (lanes of gate columns finish what those eight behind them have of the up columns; the stores above came from other lanes)
    if (MOE && act_now) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const int n_act = (lh ? late.k.N >> 1 : 0) + 64 * cp + 16 * wsel + (lc & 31);
    const uint32_t* b_late = late.k.B;
    if constexpr (MOE) b_late += late.k.expert_ids[mt] * late.k.b_estride;
#pragma unroll 1
    for (int r0 = m0 * 16; r0 < rows; r0 += 64) {
      uint32_t f = 0;
#pragma unroll 8
      for (int gi = gb0; gi < ge0; ++gi) f |= flags[(int64_t)gi * late.rows + min(r0 + lane, rows - 1)];
      uint64_t hit = __ballot(r0 + lane < rows && (f >> 16 & 1u) != 0) & 0x1111111111111111ull << (lane >> 4);
#pragma unroll 1
      for (; hit; hit &= hit - 1) {
        const int r = r0 + __builtin_ctzll(hit);
        const f32x4 v = x8_infinite_row<ZP, CHANNEL>(a_row(r), flags + r, late.rows, gb0, ge0, b_late, Sc, late.k.Z, late.k.N, late.k.group_shift,
                                                     act ? n_act : col_ok ? ncol : n_in);
        if (MOE && act_now) {
          f32x4 w;
#pragma unroll
          for (int q = 0; q < 4; ++q) w[q] = __shfl(v[q], (lane + 8) & 63);
          // (ac, ocol and their constants are those of lanes 0 .. 7)
          if (lh == 0) finish_act(r, v, w);
        } else if (col_ok) {
          finish(r, v);
        }
      }
    }
  }
}

template <bool ZP, bool CHANNEL, int MB, int KS, int WN>
__global__ __launch_bounds__(64 * KS * WN, 2) void x8_kernel(const X8Params xp) {
  x8_tile<ZP, CHANNEL, MB, KS, WN, false>(xp);
}
template <bool CHANNEL>
__global__ __launch_bounds__(512, 2) void x8_moe_kernel(const X8Params xp) {
  x8_tile<false, CHANNEL, 8, 1, 8, false, true>(xp);
}
template <bool CHANNEL>
__global__ __launch_bounds__(512, 2) void x8_prepared_kernel(const X8Params xp) {
  x8_tile<true, CHANNEL, 8, 1, 8, true>(xp);
}

// Prepared weights: the e4m3 numbers (q - z) * 2^-6 in the order in which a wavefront takes its operands: [K / 128][unit of 64 columns][16-byte
// piece 8][lane][16 bytes].  A wavefront: the two units of a column pair in one step.
__global__ __launch_bounds__(256) void x8_weights_kernel(const uint32_t* B, const uint32_t* Z, int N, int group_shift, bool channel, unsigned char* w8) {
  __shared__ __align__(16) uint32_t tables[X8_TABLES / 4];
  const int t = threadIdx.x, lane = t & 63, c = lane & 7, h = (lane >> 3) & 1, g = lane >> 4;
  if (t < X8_TABLES / 4) tables[t] = x8_table(t >> 2, t & 3);
  __syncthreads();
  const int cp = blockIdx.x * 4 + (t >> 6), step = blockIdx.y;
  if (cp * 128 >= N) return;
  const int nt = (2 * cp + h) * 64 < N ? 2 * cp + h : 2 * cp;
  u32x4 x[8];
#pragma unroll
  for (int kt = 0; kt < 8; ++kt) x[kt] = __builtin_nontemporal_load((const u32x4*)(B + (int64_t)(step * 8 + kt) * (2 * N) + nt * 128 + (4 * c + g) * 4));
  const uint32_t z = Z[(int64_t)(channel ? 0 : (4 * step) >> group_shift) * (N >> 3) + nt * 8 + c];
  unsigned char* out = w8 + step * x8_weight_step(N) + cp * 16384 + lane * 16;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const u32x4 t0 = *(const u32x4*)(tables + (z >> (4 * w) & 15u) * 4), t1 = *(const u32x4*)(tables + (z >> (4 * w + 16) & 15u) * 4);
    i32x8 o[2];
#pragma unroll
    for (int kt = 0; kt < 8; ++kt) {
      int o0, o1;
      x8_weights(x[kt][w], t0, t1, o0, o1);
      o[0][kt] = o0, o[1][kt] = o1;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int q = 0; q < 2; ++q)
        *(u32x4*)(out + (w >> 1) * 8192 + ((2 * (w & 1) + i) * 2 + q) * 1024) =
            u32x4{(uint32_t)o[i][4 * q], (uint32_t)o[i][4 * q + 1], (uint32_t)o[i][4 * q + 2], (uint32_t)o[i][4 * q + 3]};
  }
}

// Second pass of a launch with K also split across workgroups: adds the fp32 partial tiles in split order.
template <bool CHANNEL>
__global__ __launch_bounds__(256) void x8_reduce_kernel(const KParams p, int bm, int bn) {
  const int mtiles = (p.M + bm - 1) / bm;
  const int64_t piece = (int64_t)blockIdx.x * 256 + threadIdx.x;  // four columns of a row
  const int per_row = p.N >> 2;
  const int row = (int)(piece / per_row), n = (int)(piece - (int64_t)row * per_row) * 4;
  if (row >= p.M) return;
  const int mt = row / bm, strip = n / bn;
  const float* src = p.ctmp + (((int64_t)(strip * mtiles + mt) * p.splits) * bm + (row - mt * bm)) * bn + (n - strip * bn);
  f32x4 v = {0, 0, 0, 0};
  for (int s0 = 0; s0 < p.splits; s0 += 4) {
    f32x4 a[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) a[q] = *(const f32x4*)(src + (int64_t)min(s0 + q, p.splits - 1) * bm * bn);
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (s0 + q < p.splits) v += a[q];
  }
  const int base = n & ~31, cl = n & 31;
  const uint16_t* Sc = (const uint16_t*)p.S;
  const uint16_t* bias = (const uint16_t*)p.bias;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (CHANNEL) v[q] *= bf16_lo_f32(Sc[base + single_perm_pos(cl + q)]);
    if (bias) v[q] += bf16_lo_f32(bias[base + single_perm_pos(cl + q)]);
  }
  store_row4<DT_BF16, false>(p, row, n, v);
}

typedef void (*x8_fn)(const X8Params);
template <int MB, int KS, int WN>
static x8_fn pick_x8(bool zp, bool channel) {
  if (zp) return channel ? x8_kernel<true, true, MB, KS, WN> : x8_kernel<true, false, MB, KS, WN>;
  return channel ? x8_kernel<false, true, MB, KS, WN> : x8_kernel<false, false, MB, KS, WN>;
}

int64_t x8_scratch_bytes(int64_t rows, int64_t k) {
  const int64_t r = x8_rows(rows), g = k / X8_G;
  return r * g * 256 + (r * g * 4 + 255) / 256 * 256;
}

int64_t x8_weight_bytes(int64_t k, int64_t n) { return k / X8_G * x8_weight_step(n); }

static x8_fn pick_x8_shape(int mb, int ks, int tn, bool zp, bool channel, bool prep) {
  if (prep) return ks != 1 || mb != 8 || tn != 512 || !zp ? nullptr : channel ? x8_prepared_kernel<true> : x8_prepared_kernel<false>;
  if (ks == 1 && mb == 8) return tn == 512 ? pick_x8<8, 1, 8>(zp, channel) : tn == 256 ? pick_x8<8, 1, 4>(zp, channel) : nullptr;
  if (ks != 2 || tn != 256) return nullptr;
  switch (mb) {
    case 8: return pick_x8<8, 2, 4>(zp, channel);
    case 7: return pick_x8<7, 2, 4>(zp, channel);
    case 6: return pick_x8<6, 2, 4>(zp, channel);
    case 5: return pick_x8<5, 2, 4>(zp, channel);
    default: return nullptr;
  }
}

int launch_x8(const w4a16_gemm_args* a, const Plan& pl, void* scratch, hipStream_t stream) {
  const bool zp = a->b_zeros != nullptr, channel = pl.gm == GM_CHANNEL, prep = pl.kind == 7;
  const x8_fn fn = pick_x8_shape(pl.mb, pl.ks, pl.tn, zp, channel, prep);
  if (!fn || a->dtype != DT_BF16 || (a->wtype != W4A16_WTYPE_U4B8 && a->wtype != W4A16_WTYPE_U4) ||
      (a->flags & (W4A16_F_ZP_FLOAT | W4A16_F_MOE)) || pl.gm == GM_GIDX || pl.use_perm || pl.splits < 1 || pl.kps % 4 != 0)
    return fail(W4A16_EINVAL, "unsupported kernel variant");
  if (pl.tiles <= 0) return 0;
  X8Params xp;
  xp.k = make_kparams(a, pl);
  const int groups = (int)(a->size_k / X8_G);
  const int64_t r = x8_rows(a->size_m);
  unsigned char* base = (unsigned char*)scratch;
  xp.rec = base;
  xp.scl = (const uint32_t*)(base + r * groups * 256);
  xp.rows = (int)r;
  xp.w8 = nullptr;
  if (prep) {
    unsigned char* w8 = base + x8_scratch_bytes(a->size_m, a->size_k);
    xp.w8 = w8;
    hipLaunchKernelGGL(x8_weights_kernel, dim3((unsigned)ceil_div(a->size_n, 512), (unsigned)groups), dim3(256), 0,
                       stream, xp.k.B, xp.k.Z, xp.k.N, xp.k.group_shift, channel, w8);
    W4A16_HIP(hipGetLastError());
  }
  // (the rows of the tiles, a multiple of 16 that is at most M + 127: never more than x8_rows)
  const int64_t blocks = (int64_t)pl.mtiles * pl.bm / 16;
  // (steps per workgroup: few rows fill the chip only with one.  40 problems of 167 to 1562 rows for which x8_rows would ask for four and the tiles'
  //  rows ask for one: one 0.983 of the time in the mean, at worst 1.00)
  const int sg = blocks * groups >= 16 * num_cus() ? 4 : 1;
  hipLaunchKernelGGL((sg == 4 ? x8_split_kernel<4> : x8_split_kernel<1>), dim3((unsigned)blocks, (unsigned)ceil_div(groups, sg)), dim3(256), 0,
                     stream, (const uint16_t*)a->a, a->lda, (int)a->size_m, (int)r, groups, (unsigned char*)xp.rec,
                     (uint32_t*)xp.scl);
  W4A16_HIP(hipGetLastError());
  const int smem = x8_smem(pl.mb, pl.ks, pl.tn / 64) + (zp ? X8_TABLES : 0);
  W4A16_HIP(allow_dynamic_lds((const void*)fn, smem));
  hipLaunchKernelGGL(fn, dim3((unsigned)((int64_t)pl.tiles * pl.splits)), dim3((unsigned)(pl.ks * pl.tn)), smem, stream, xp);
  W4A16_HIP(hipGetLastError());
  if (pl.splits > 1) {
    const dim3 n((unsigned)ceil_div(a->size_m * (a->size_n / 4), 256));
    if (channel)
      hipLaunchKernelGGL(x8_reduce_kernel<true>, n, dim3(256), 0, stream, xp.k, pl.bm, pl.tn);
    else
      hipLaunchKernelGGL(x8_reduce_kernel<false>, n, dim3(256), 0, stream, xp.k, pl.bm, pl.tn);
    W4A16_HIP(hipGetLastError());
  }
  return 0;
}

int64_t x8_moe_scratch_bytes(int64_t n_sorted, int64_t k) {
  const int64_t r = (n_sorted + 127) / 128 * 128, g = k / X8_G;
  return r * g * 256 + (r * g * 4 + 255) / 256 * 256;
}

// MoE blocks of 128 slots, uint4b8: the prefill kernel's tiles, plan and second pass
int launch_x8_moe(const w4a16_gemm_args* a, const Plan& pl, void* scratch, hipStream_t stream) {
  const bool channel = pl.gm == GM_CHANNEL;
  if (a->dtype != DT_BF16 || a->wtype != W4A16_WTYPE_U4B8 || !(a->flags & W4A16_F_MOE) || pl.gm == GM_GIDX || pl.bm != 128 || pl.tn != 512 ||
      pl.splits != 1 || pl.dyn_slots <= 0 || pl.total_ksteps % 4 != 0 || (!channel && pl.group_ksteps % 4 != 0))
    return fail(W4A16_EINVAL, "unsupported kernel variant");
  if (pl.tiles <= 0) return 0;
  X8Params xp{};
  xp.k = make_kparams(a, pl);
  const int groups = (int)(a->size_k / X8_G), rows = pl.mtiles * 128;
  unsigned char* base = (unsigned char*)scratch;
  xp.rec = base;
  xp.scl = (const uint32_t*)(base + (int64_t)rows * groups * 256);
  xp.rows = rows;
  const X8Slots slots = {xp.k.sorted_ids, xp.k.ntpp, xp.k.n_sorted, xp.k.c_rows, xp.k.top_k, xp.k.a_by_slot};
  hipLaunchKernelGGL(x8_split_slots_kernel, dim3((unsigned)(rows / 16), (unsigned)ceil_div(groups, 4)), dim3(256), 0, stream, (const uint16_t*)a->a, a->lda,
                     rows, groups, base, (uint32_t*)xp.scl, slots);
  W4A16_HIP(hipGetLastError());
  const x8_fn fn = channel ? x8_moe_kernel<true> : x8_moe_kernel<false>;
  const int smem = x8_smem(8, 1, 8) + 128 * 8;
  W4A16_HIP(allow_dynamic_lds((const void*)fn, smem));
  hipLaunchKernelGGL(fn, dim3((unsigned)(pl.tiles + mid_tail_pieces(pl.tiles, pl.dyn_slots))), dim3(512), smem, stream, xp);
  W4A16_HIP(hipGetLastError());
  return launch_fat_reduce(a, pl, xp.k, stream);
}

}  // namespace w4a16
