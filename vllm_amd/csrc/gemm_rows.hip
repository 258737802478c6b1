// W4A16 GEMM for gfx950, 17 and more rows on tiles of 32 or 48 rows x 64 columns with the arithmetic of the 16-row kernel (gemm_decode.hip): integer
// weights go to the MFMA unscaled, offset and scale are applied to the fp32 sums once per group, so no weight is rounded.  That kernel reads and converts
// a weight strip once per 16 rows; here every converted operand feeds two or three MFMAs, and the strip is streamed once.
//
//   workgroup  eight wavefronts cut the split's K range into contiguous parts of whole stages (two k-steps, 64 K rows), as in the 16-row kernel: weights and
//              activations two stages ahead in registers, activations bounced through wavefront-private LDS into operand order, an LDS sum of the
//              wavefronts' tiles, an ordered cross-workgroup sum behind an arrival counter (see store_coherent2).
//   64 columns  a tile of 48 x 64 holds 48 sums, 48 products of the group and 12 row sums; of 128 columns they alone would fill the registers.
// Requirements (host-checked): dense, integer 4-bit weights, K % 128 == 0, groups of 128 rows x a power of two or one scale per column, A's columns in
// weight order.
#include <type_traits>

#include "gemm_kernels.h"

namespace w4a16 {

constexpr int RW_NW = 8;      // wavefronts
constexpr int RW_TN = 64;
constexpr int RW_RS = 84;     // floats per row of a reduction slab (4 mod 16)
constexpr int RW_AROW = 36;   // dwords per row of an activation slab: 32 and 4 (bank = 36 row + 4 piece + dword: conflict-free)
constexpr int rw_smem(int mb) {
  const int sums = RW_NW * mb * 16 * RW_RS * 4, slabs = RW_NW * mb * 16 * RW_AROW * 4;
  return sums > slabs ? sums : slabs;
}

template <int DT, bool ZP, bool CHANNEL, int MB>
__global__ __launch_bounds__(RW_NW * 64, 2) void rows_kernel(const KParams p) {
  constexpr bool HI_TRICK = DT == DT_F16 && !ZP;
  constexpr int BM = 16 * MB, NW = RW_NW;
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ int s_last;
  const int t = threadIdx.x, lane = t & 63;
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int c = lane & 7, h = (lane >> 3) & 1, g = lane >> 4;

  // (the splits of a tile: x; tiles of consecutive workgroups walk M first, so those that share a strip run together)
  const int mtiles = (p.M + BM - 1) / BM;
  int tile, split;
  if (p.xcd_map) {  // all splits of a tile on one XCD
    tile = blockIdx.z * 8 + blockIdx.x, split = blockIdx.y;
  } else {
    tile = blockIdx.y, split = blockIdx.x;
  }
  const int ct = tile / mtiles, mt = tile - ct * mtiles, row0 = mt * BM;

  const uint16_t* Sc = (const uint16_t*)p.S;
  const uint16_t* bias = (const uint16_t*)p.bias;
  // activation loads: lane -> row (lane >> 3) + 8 i, 16-byte piece (lane & 7) of the stage's 128 bytes (the last row in place of those behind it)
  const int ar = lane >> 3, ap = lane & 7;
  const char* abase = (const char*)p.A + (int64_t)row0 * p.lda * 2;
  uint32_t aoff[2 * MB];
#pragma unroll
  for (int i = 0; i < 2 * MB; ++i) aoff[i] = (uint32_t)min(ar + 8 * i, p.M - 1 - row0) * ((uint32_t)p.lda * 2) + ap * 16;  // (the host checks the size)

  // ---- this wavefront's units of 128 K rows (two stages, one fold)
  const int un_b = split * p.ksteps_per_split / 4, un_e = min(un_b + p.ksteps_per_split / 4, p.total_ksteps / 4);
  const int w_b = un_b + (un_e - un_b) * wv / NW, w_e = un_b + (un_e - un_b) * (wv + 1) / NW;

  const int64_t b_row = p.N * 2;  // words per k-tile row
  const uint32_t* bp = p.B + (int64_t)ct * 128 + (4 * c + g) * 4 + 2 * h;
  const uint16_t* sp = Sc + (int64_t)ct * 64 + 8 * c + 4 * h;
  const uint32_t* zp = ZP ? p.Z + ct * 8 + c : nullptr;

  uint32_t* slab = (uint32_t*)smem + wv * (BM * RW_AROW);
  uint32_t* slab_wr = slab + ar * RW_AROW + ap * 4;
  const uint32_t* slab_rd = slab + (lane & 15) * RW_AROW + g;

  struct Stage {
    u32x2 b[4];
    u32x4 a[2 * MB];
  };
  Stage st[2];
  u32x2 sc = {0, 0}, sc_next = {0, 0};
  uint32_t zq = 0, zq_next = 0;
  // (indices are clamped instead of guarded: the last unit is read again, which keeps the loop free of branches)
  auto issue = [&](Stage& s, int unit, int half) {
    const int sidx = 2 * min(unit, w_e - 1) + half;
#pragma unroll
    for (int i = 0; i < 2 * MB; ++i) s.a[i] = *(const u32x4*)(abase + (int64_t)sidx * 128 + aoff[i]);
#pragma unroll
    for (int i = 0; i < 4; ++i) s.b[i] = __builtin_nontemporal_load((const u32x2*)(bp + (4 * sidx + i) * b_row));
  };
  auto issue_scales = [&](int unit) {
    const int64_t gi = CHANNEL ? 0 : (4 * min(unit, w_e - 1)) >> p.group_shift;
    if (!CHANNEL) sc_next = *(const u32x2*)(sp + gi * p.N);
    if (ZP) zq_next = zp[gi * (p.N >> 3)];
  };

  f32x4 acc[MB][2][2], tmp[MB][2][2], rs[MB];
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[m][i >> 1][i & 1] = f32x4{0, 0, 0, 0};

  // acc += s * (tmp - e * rs),  e = E + z  (HI_TRICK: the bias operand already carries E + 8, e = 1)
  auto fold = [&]() {
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        const float s = CHANNEL ? 1.f : hf ? hi_f32<DT>(sc[w]) : lo_f32<DT>(sc[w]);
        float e = 1.f;
        if constexpr (!HI_TRICK) e = (DT == DT_F16 ? 1024.f : 128.f) + (ZP ? (float)((zq >> (4 * (2 * h + w) + 16 * hf)) & 0xf) : 8.f);
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[m][w][hf][r] = __builtin_fmaf(s, __builtin_fmaf(-e, rs[m][r], tmp[m][w][hf][r]), acc[m][w][hf][r]);
      }
  };
  auto consume = [&](const Stage& s, auto first_tag) __attribute__((always_inline)) {
    // activations: rows of 128 bytes in, MFMA operands (row, K pairs 8 s + 2 g) out
#pragma unroll
    for (int i = 0; i < 2 * MB; ++i) *(u32x4*)(slab_wr + 8 * i * RW_AROW) = s.a[i];
    lds_lanes_in_order();
    u32x4 vb;  // operand of the row sums
    if constexpr (HI_TRICK) {
      vb = u32x4{RAW_BIAS_LO, RAW_BIAS_HI, RAW_BIAS_LO, RAW_BIAS_HI};
    } else {
      const uint32_t one = DT == DT_F16 ? 0x3c003c00u : 0x3f803f80u;
      vb = u32x4{one, one, one, one};
    }
    const f32x4 zero = {0, 0, 0, 0};
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      u32x4 af[MB], o[2][2];
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        const uint32_t* q = slab_rd + 16 * m * RW_AROW + kk * 16;
        af[m] = u32x4{q[0], q[4], q[8], q[12]};
      }
#pragma unroll
      for (int w = 0; w < 2; ++w) raw_pair<DT, HI_TRICK>(s.b[2 * kk][w], s.b[2 * kk + 1][w], o[w][0], o[w][1]);
      const bool first = decltype(first_tag)::value && kk == 0;
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        rs[m] = mfma16x16x32<DT>(af[m], vb, first ? zero : rs[m]);
#pragma unroll
        for (int i = 0; i < 4; ++i) tmp[m][i >> 1][i & 1] = mfma16x16x32<DT>(af[m], o[i >> 1][i & 1], first ? zero : tmp[m][i >> 1][i & 1]);
      }
    }
  };

  if (w_b < w_e) {
    issue_scales(w_b);
    issue(st[0], w_b, 0);
    issue(st[1], w_b, 1);
    Pace pace;
    pace.start(w_e - w_b);
#pragma unroll 1
    for (int unit = w_b; unit < w_e; ++unit) {
      pace.round(unit - w_b);
      sc = sc_next, zq = zq_next;
      issue_scales(unit + 1);
      __builtin_amdgcn_sched_barrier(0);
      consume(st[0], std::true_type{});
      __builtin_amdgcn_sched_barrier(0);
      issue(st[0], unit + 1, 0);
      __builtin_amdgcn_sched_barrier(0);
      consume(st[1], std::false_type{});
      __builtin_amdgcn_sched_barrier(0);
      issue(st[1], unit + 1, 1);
      __builtin_amdgcn_sched_barrier(0);
      fold();
    }
  }

  // ------------------------------------------------------------------------------ epilogue
  // red[wavefront][row][RW_RS floats]: column 32 h + 16 w + 8 half + c at 40 h + 16 w + 8 half + c
  float* red = (float*)smem;
  constexpr int RPP = NW * 2, NP = BM / RPP;  // 32 threads to a row: rows per pass, passes
  const int fr0 = t >> 5, fc = (t & 31) * 2, fpos = fc + (fc >= 32 ? 8 : 0);
  const int ncol = ct * RW_TN + fc;
  float cs[2] = {1.f, 1.f}, bs[2] = {0.f, 0.f};
  {
    const int base = ncol & ~31, cl = ncol & 31;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if (CHANNEL) cs[j] = lo_f32<DT>(Sc[base + single_perm_pos(cl + j)]);
      if (bias) bs[j] = lo_f32<DT>(bias[base + single_perm_pos(cl + j)]);
    }
  }
  __syncthreads();  // activation slabs no longer read
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[(wv * BM + 16 * m + 4 * g + r) * RW_RS + 40 * h + 8 * i + c] = acc[m][i >> 1][i & 1][r];
  __syncthreads();
  float v[NP][2];
#pragma unroll
  for (int ps = 0; ps < NP; ++ps) {
    v[ps][0] = v[ps][1] = 0.f;
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) {
      const float* src = red + (ww * BM + fr0 + RPP * ps) * RW_RS + fpos;
      v[ps][0] += src[0], v[ps][1] += src[1];
    }
  }
  auto finish = [&](int ps) {
    const int row = row0 + fr0 + RPP * ps;
    if (row >= p.M) return;
    *(uint32_t*)((uint16_t*)p.C + (int64_t)row * p.N + ncol) = pack2<DT>(v[ps][0] * cs[0] + bs[0], v[ps][1] * cs[1] + bs[1]);
  };
  if (p.splits == 1) {
#pragma unroll
    for (int ps = 0; ps < NP; ++ps) finish(ps);
    return;
  }
  float* const parts = p.ctmp + (int64_t)tile * p.splits * (BM * RW_TN) + fr0 * RW_TN + fc;
#pragma unroll
  for (int ps = 0; ps < NP; ++ps)
    if (row0 + fr0 + RPP * ps < p.M) store_coherent2(parts + (split * BM + RPP * ps) * RW_TN, v[ps][0], v[ps][1]);
  // ---- the last split to arrive sums all partial tiles in split order
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (t == 0) s_last = arrive_last(p.locks + tile * p.lock_stride, p.splits);
  __syncthreads();
  if (!s_last) return;
#pragma unroll
  for (int ps = 0; ps < NP; ++ps) v[ps][0] = v[ps][1] = 0.f;
  // (four splits' loads are in flight together)
  for (int s0 = 0; s0 < p.splits; s0 += 4) {
    float a[NP][4][2];
#pragma unroll
    for (int ps = 0; ps < NP; ++ps)
#pragma unroll
      for (int i = 0; i < 4; ++i) load_coherent2(parts + (min(s0 + i, p.splits - 1) * BM + RPP * ps) * RW_TN, a[ps][i][0], a[ps][i][1]);
#pragma unroll
    for (int ps = 0; ps < NP; ++ps)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (s0 + i < p.splits) v[ps][0] += a[ps][i][0], v[ps][1] += a[ps][i][1];
  }
#pragma unroll
  for (int ps = 0; ps < NP; ++ps) finish(ps);
}

typedef void (*rows_fn)(const KParams);
template <int DT, int MB>
static rows_fn pick_rows(bool zp, bool channel) {
  if (zp) return channel ? rows_kernel<DT, true, true, MB> : rows_kernel<DT, true, false, MB>;
  return channel ? rows_kernel<DT, false, true, MB> : rows_kernel<DT, false, false, MB>;
}
template <int DT>
static rows_fn pick_rows(int mb, bool zp, bool channel) {
  return mb == 2 ? pick_rows<DT, 2>(zp, channel) : mb == 3 ? pick_rows<DT, 3>(zp, channel) : nullptr;
}

int launch_rows(const w4a16_gemm_args* a, const Plan& pl, hipStream_t stream) {
  const bool zp = a->b_zeros != nullptr, channel = pl.gm == GM_CHANNEL;
  const rows_fn fn = a->dtype == DT_F16 ? pick_rows<DT_F16>(pl.mb, zp, channel) : pick_rows<DT_BF16>(pl.mb, zp, channel);
  if (!fn || (a->wtype != W4A16_WTYPE_U4B8 && a->wtype != W4A16_WTYPE_U4) || (a->flags & (W4A16_F_ZP_FLOAT | W4A16_F_MOE)) || pl.gm == GM_GIDX || pl.use_perm ||
      pl.tn != RW_TN || pl.total_ksteps % 4 != 0 || pl.kps % 4 != 0 || pl.splits < 1 || (int64_t)pl.kps * pl.splits < pl.total_ksteps ||
      (!channel && (pl.group_ksteps % 4 != 0 || (pl.group_ksteps & (pl.group_ksteps - 1)) != 0)) || a->lda < 0 || a->lda * 2 * pl.bm >= (1LL << 31) ||
      (pl.xcd_map && pl.tiles % 8 != 0) || pl.tiles > 65535)
    return fail(W4A16_EINVAL, "unsupported kernel variant");
  if (pl.tiles <= 0) return 0;
  const KParams p = make_kparams(a, pl);
  const int smem = rw_smem(pl.mb);
  W4A16_HIP(allow_dynamic_lds((const void*)fn, smem));
  const dim3 grid = pl.xcd_map ? dim3(8, (unsigned)pl.splits, (unsigned)(pl.tiles / 8)) : dim3((unsigned)pl.splits, (unsigned)pl.tiles);
  hipLaunchKernelGGL(fn, grid, dim3(RW_NW * 64), smem, stream, p);
  W4A16_HIP(hipGetLastError());
  return 0;
}

}  // namespace w4a16
