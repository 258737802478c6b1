// W4A16 prefill GEMM for gfx950 (large M): C[M,N] = A[M,K] * dequant(Bq)[K,N] (+bias).
//
// Same operand layouts as the skinny kernel (gemm_common.h), tiled for the matrix cores:
//   workgroup tile 128 rows x 512 columns, 4 wavefronts, each owning 128 rows x 128 columns (one column
//   pair): 8 m-blocks x 8 MFMA column groups = 64 v_mfma_f32_16x16x32 per k-step, 256 fp32 accumulators
//   per lane (one wavefront per SIMD, 512 registers).
//   weights      each wavefront streams its own column pair global -> registers (128-bit loads) and
//                dequantises it once per k-step (scale applied per element, so the B operand equals the
//                reference's half(q - z) * half(s)); every dequantised operand feeds 8 MFMAs.
//   activations  the workgroup stages 128 rows x 64 K (two k-steps, 128 contiguous bytes per row) into LDS,
//                double buffered, already in MFMA fragment order, so an A operand is one conflict-free
//                ds_read_b128; one barrier per two k-steps (128 MFMAs per wavefront).
// MFMA work per byte of weights is 64x the decode kernel's; the bound is the matrix pipe, and the VALU work
// of dequantisation (about 105 instructions per 64 MFMAs for fp16) is interleaved with them: the MFMAs run
// word-major (16 per Marlin word), and as soon as a word's operands are dead the next k-step's word is
// dequantised into the same registers.  One wavefront per SIMD has nothing to hide a wait behind, so (1) the A operands of a k-step are
// read from LDS during the last word of the one before; (2) a register's three dependent steps stand between three MFMA pairs; (3) scales and
// zero points of groups of 128 rows and more come once per 128 rows (ONCE), shorter groups have a loop of their own: with both loops in one
// kernel the registers did not reach.  Dense 4096 x 28672 and 5120 x 13824, 512 to 4096 rows: groups of 32 and 64 0.92 - 0.98 of the time (fp16
// uint4b8, 1501 rows: 337 -> 323 us), of 128 0.98 - 1.00, channel-wise level; MoE blocks of 128, three expert shapes: 0.98 in the mean, short
// groups 0.96.
// MoE blocks of 128 sorted slots run here too when experts are large and full (_tall_from in fused_marlin_moe.py): the 64-row kernel dequantises
// every weight once per 64 rows (8 experts of 4096 x 14336, top-2, 4096 tokens, bf16: GEMM1 2129 -> 1815 us, GEMM2 1011 -> 874).
// Requirements (host-checked; otherwise the skinny kernel runs): K % 128 == 0, no per-row g_idx.
#include <type_traits>

#include "gemm_kernels.h"

namespace w4a16 {

constexpr int FB_MB = 8;     // m-blocks per wavefront
constexpr int FB_D = 4;      // weight k-steps in flight per wavefront
constexpr int FB_ABUF = 2 * FB_MB * 64 * 16;  // bytes of one A buffer: 2 k-steps x 8 m-blocks x 64 lanes x 16 B
constexpr int FB_SLABS = 4 * 16 * RED_RS * 4;                // four wavefront slabs of the epilogue
constexpr int FB_SMEM = (2 * FB_ABUF > FB_SLABS ? 2 * FB_ABUF : FB_SLABS) + FB_BM * 8;  // + C row and routing weight of each tile row

// BITS = 8: uint8b128 or (FP8) float8_e4m3fn weights in the 8-bit Marlin layout: twice the words per lane, the same 64
// MFMAs per k-step; no zero points.
// FP4 = 1 / 2: float4_e2m1f weights (4-bit layout) with NVFP4 / MXFP4 scale records, one 16-byte record per lane and
// k-step / two k-steps (the host sets the group to 1 / 2 k-steps); NVFP4's global scale is applied to the accumulator.
// ZPF: uint4 weights with fp16 zero points laid out like the scales (HQQ): operand = fma(q, s, -half(zp * s)).
// ONCE: integer 4-bit weights with groups of 128 rows at least, or one scale per column.
// MOE: blocks of 128 sorted token slots (integer 4-bit weights); rows are gathered through sorted_token_ids while staging.
template <int DT, bool ZP, bool CHANNEL, int BITS = 4, bool FP8 = false, int FP4 = 0, bool ZPF = false, bool MOE = false, bool ONCE = false>
__global__ __launch_bounds__(256) void fat_kernel(const KParams p) {
  static_assert(!ZPF || (DT == DT_F16 && !ZP && !CHANNEL && BITS == 4 && FP4 == 0), "float zero points: fp16 uint4 grouped");
  static_assert(BITS == 4 || (BITS == 8 && !ZP), "8-bit weights have no zero points");
  static_assert(!FP8 || BITS == 8, "fp8 weights use the 8-bit layout");
  static_assert(FP4 == 0 || (BITS == 4 && !ZP && !CHANNEL), "fp4 weights: grouped scale records, no zero points");
  static_assert(!MOE || (BITS == 4 && FP4 == 0 && !ZPF), "MoE: integer 4-bit weights");
  constexpr bool UNIT = CHANNEL;
  extern __shared__ __align__(16) unsigned char smem[];
  int* s_crow = (int*)(smem + FB_SMEM - FB_BM * 8);
  float* s_tw = (float*)(smem + FB_SMEM - FB_BM * 4);
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int c = lane & 7, h = (lane >> 3) & 1, g = lane >> 4;

  // tile order: M first, so workgroups resident together share weight strips (MoE: neighbouring blocks mostly belong to
  // the same expert)
  int mtiles = MOE ? (p.n_sorted + FB_BM - 1) / FB_BM : (p.M + FB_BM - 1) / FB_BM;
  int ks_b = 0, ks_e = p.total_ksteps, split = 0, nsplit = 1, part = 0;
  int j = blockIdx.x;
  if constexpr (MOE) {
    zero_fill_side_job(p);
    mtiles = min((*p.ntpp + FB_BM - 1) / FB_BM, mtiles);
    if (mtiles == 0) return;
    // live tiles; those of the last, partly filled round in K pieces (see tail_split), which walk the tiles first, then K
    const TailSplit d = tail_split(mtiles * p.ncp, p.dyn_slots, p.total_ksteps, FB_MIN_SPLIT);
    if (j < d.F) {
      // workgroup b runs on XCD b mod 8: every XCD gets a contiguous run of tiles, so that the ones it holds at a time share
      // their expert's weight strips and activation rows in its L2
      if ((d.F & 7) == 0) j = (j & 7) * (d.F >> 3) + (j >> 3);
    } else {
      const int u = j - d.F;
      if (u >= d.R * d.S) return;
      part = u % d.R, split = u / d.R, nsplit = d.S;
      ks_b = split * d.kps, ks_e = min(ks_b + d.kps, p.total_ksteps);
      j = d.F + part;
    }
  }
  int mt = j % mtiles, nt4 = j / mtiles;
  if (MOE) chunked_tile(j, mtiles, p.ncp, mt, nt4);
  const int cp = nt4 * 4 + wv;                 // column pair of this wavefront
  const bool wave_on = cp * 128 < p.N;         // N not a multiple of 512: trailing wavefronts only help staging
  const int row0 = mt * FB_BM;

  const uint32_t* Bq = p.B;
  const uint16_t* Sc = (const uint16_t*)p.S;
  const uint32_t* Zp = p.Z;
  const uint16_t* bias = (const uint16_t*)p.bias;
  if constexpr (MOE) {
    const int e = p.expert_ids[mt];
    if (e < 0) return;  // expert of another rank
    Bq += e * p.b_estride;
    Sc += e * p.s_estride;
    if (ZP) Zp += e * p.z_estride;
    if (bias) bias += e * p.n_estride;
  }
  // which A row feeds tile row r and which C row receives it (-1: none)
  auto tile_row_ids = [&](int r, int& src, int& dst) {
    src = dst = -1;
    const int id = p.sorted_ids[row0 + r];
    if ((unsigned)id < (unsigned)p.c_rows) {
      src = p.a_by_slot ? row0 + r : id / p.top_k;
      dst = id;
    }
  };
  if (MOE && t < FB_BM) {
    int src, dst;
    tile_row_ids(t, src, dst);
    s_crow[t] = dst;
    if (p.mul_topk) s_tw[t] = dst >= 0 ? p.topk_w[dst] : 0.f;
  }

  // ---- weights of this wavefront
  // (fused SiLU-and-mul: gate n-tile cp paired with the up n-tile of the same output columns, N/128 + cp)
  const int nt = !wave_on ? 0 : (MOE && p.act) ? (h ? (p.N >> 7) + cp : cp) : ((2 * cp + h) * 64 < p.N ? 2 * cp + h : 0);
  // 4-bit: 32 u32x4 per n-tile and k-tile, one per Marlin thread; 8-bit: 64, two per thread (words 2w + half)
  const int64_t b_row = (BITS == 4) ? (p.N >> 1) : p.N;
  const u32x4* bp = (const u32x4*)Bq + nt * (8 * BITS) + (4 * c + g) * (BITS / 4);
  const int64_t s_row = p.N >> 3;
  const u32x4* sp = (const u32x4*)Sc + nt * 8 + c;
  const uint32_t* zp = ZP ? Zp + nt * 8 + c : nullptr;
  const u32x4* zfp = ZPF ? (const u32x4*)p.Z + nt * 8 + c : nullptr;  // fp16 zero points: indexed like the scales

  // ---- activation staging: thread t loads piece (t & 7) of rows (t >> 3) + 32 i, i = 0..3
  const int piece = t & 7;
  const uint16_t* arow[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    int r = row0 + (t >> 3) + 32 * i;
    if constexpr (MOE) {
      int dst;
      tile_row_ids((t >> 3) + 32 * i, r, dst);
      if (r < 0) r = 0;  // slots without a token read row 0; never stored
    } else if (r >= p.M) {
      r = p.M - 1;  // rows past the end replicate the last row; never stored
    }
    arow[i] = (const uint16_t*)p.A + (int64_t)r * p.lda + piece * 8;
  }
  // LDS A layout: [buffer][k-step 2][m-block 8][lane 64][4 dwords]; the 16 bytes of (row, piece) are the K
  // pairs 8*pp + 2q (pp = piece & 3), which belong to lane (q*16 + row%16), dword pp, of k-step piece >> 2.
  uint32_t* lds = (uint32_t*)smem;
  int a_wr[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = (t >> 3) + 32 * i;
    a_wr[i] = (((piece >> 2) * FB_MB + (r >> 4)) * 64 + (r & 15)) * 4 + (piece & 3);
  }
  u32x4 areg[4];
  // (chunk and k-step indices are clamped instead of guarded: the last iteration re-reads its own data, which
  //  keeps the main loop free of branches, so the compiler can overlap LDS reads and dequantisation with MFMAs)
  auto load_a = [&](int chunk) {  // chunk, k-step: relative to ks_b
    chunk = min(ks_b / 2 + chunk, ks_e / 2 - 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) areg[i] = *(const u32x4*)(arow[i] + chunk * 64);
  };
  auto store_a = [&](int buf) {
    uint32_t* dst = lds + buf * (FB_ABUF / 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int q = 0; q < 4; ++q) dst[a_wr[i] + q * 64] = areg[i][q];
    }
  };

  struct Stage {
    u32x4 b0, b1, sc;
    u32x4 b0h, b1h;  // 8-bit weights only: the thread's words 2, 3
    u32x4 zf;        // float zero points only
    uint32_t zq;
  };
  Stage st[FB_D];
  auto issue = [&](Stage& s, int ks) {
    ks = min(ks_b + ks, ks_e - 1);
    int gi = 0;
    if (!CHANNEL && !ONCE) gi = ks >> p.group_shift;  // the host only picks this kernel for power-of-two group sizes
    if (!CHANNEL && !ONCE) s.sc = sp[(int64_t)gi * s_row];
    if (ZP && !ONCE) s.zq = zp[(int64_t)gi * s_row];
    if (FP4 == 2) s.zq = ks & 1;  // which half of the two-k-step scale record
    if (ZPF) s.zf = zfp[(int64_t)gi * s_row];
    s.b0 = bp[(int64_t)(2 * ks) * b_row];
    s.b1 = bp[(int64_t)(2 * ks + 1) * b_row];
    if constexpr (BITS == 8) {
      s.b0h = bp[(int64_t)(2 * ks) * b_row + 1];
      s.b1h = bp[(int64_t)(2 * ks + 1) * b_row + 1];
    }
  };
  // groups of 128 rows at least: scales and zero points once per loop iteration
  u32x4 sc128 = {0, 0, 0, 0};
  uint32_t zq128 = 0;
  auto issue_scales = [&](int ks) {
    const int gi = CHANNEL ? 0 : min(ks_b + ks, ks_e - 1) >> p.group_shift;
    if (!CHANNEL) sc128 = sp[(int64_t)gi * s_row];
    if (ZP) zq128 = zp[(int64_t)gi * s_row];
  };
  struct Fp4Scales { float a0, a1, b0, b1; };
  auto fp4_scales = [&](const Stage& s, int w) {
    Fp4Scales r{1.f, 1.f, 1.f, 1.f};
    if constexpr (FP4 == 1) {
      const uint32_t ba = fp4_scale_bytes(s.sc[0], s.sc[1], w), bb = fp4_scale_bytes(s.sc[2], s.sc[3], w);
      r = Fp4Scales{nvfp4_scale_f32(ba & 0xff), nvfp4_scale_f32(ba >> 16), nvfp4_scale_f32(bb & 0xff), nvfp4_scale_f32(bb >> 16)};
    } else if constexpr (FP4 == 2) {
      const uint32_t bs = s.zq ? fp4_scale_bytes(s.sc[2], s.sc[3], w) : fp4_scale_bytes(s.sc[0], s.sc[1], w);
      const float s0 = mxfp4_scale_f32(bs & 0xff), s1 = mxfp4_scale_f32(bs >> 16);
      r = Fp4Scales{s0, s1, s0, s1};
    }
    return r;
  };
  // 8-bit: the words of Marlin word position w are elements 2(w & 1) [column half 0] and 2(w & 1) + 1 [half 1] of
  // the thread's first (w < 2) or second 16 bytes, per k-tile
  auto word8 = [&](const Stage& s, int w, int ktile, int half) -> uint32_t {
    const u32x4& v = ktile == 0 ? (w < 2 ? s.b0 : s.b0h) : (w < 2 ? s.b1 : s.b1h);
    return v[2 * (w & 1) + half];
  };
  auto col_const = [&](const Stage& s, int w) {
    return make_col_const<DT, UNIT>(CHANNEL ? 0u : ONCE ? sc128[w] : s.sc[w], ZP ? zero_pair(ONCE ? zq128 : s.zq, w) : ZERO_U4B8);
  };

  f32x4 acc[FB_MB][4][2];
#pragma unroll
  for (int mb = 0; mb < FB_MB; ++mb)
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      acc[mb][w][0] = f32x4{0, 0, 0, 0};
      acc[mb][w][1] = f32x4{0, 0, 0, 0};
    }

  const int nchunks = (ks_e - ks_b) / 2;  // even: K % 128 == 0, pieces are multiples of 4 k-steps

  // ---- prologue
  load_a(0);
  if constexpr (ONCE) issue_scales(0);
#pragma unroll
  for (int j = 0; j < FB_D; ++j) issue(st[j], j);
  store_a(0);
  // B operands of the current and of the next k-step (the roles swap every k-step)
  u32x4 ob[2][4][2];
  // integer 4-bit weights: the dequantisation constants of the four word positions.  A loop iteration covers four
  // k-steps (128 rows of K), so with groups of 128 rows or more, or one scale per column, they change at most once
  // per iteration and are kept in registers instead of being rebuilt from the scale and zero-point words every k-step.
  constexpr bool CONSTS = (BITS == 4 && FP4 == 0 && !ZPF);
  ColConst<DT> ccs[4];
  if constexpr (CONSTS) {
#pragma unroll
    for (int w = 0; w < 4; ++w) ccs[w] = col_const(st[0], w);
  }
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    if constexpr (ZPF) {
      dequant_pair_zpf(st[0].b0[w], st[0].b1[w], st[0].sc[w], as_u32(as_h2(st[0].zf[w]) * as_h2(st[0].sc[w])),
                       ob[0][w][0], ob[0][w][1]);
    } else if constexpr (FP4 != 0) {
      const Fp4Scales fs = fp4_scales(st[0], w);
      dequant_pair_fp4<DT>(st[0].b0[w], st[0].b1[w], fs.a0, fs.a1, fs.b0, fs.b1, ob[0][w][0], ob[0][w][1]);
    } else if constexpr (BITS == 4) {
      dequant_pair<DT, UNIT>(st[0].b0[w], st[0].b1[w], ccs[w], ob[0][w][0], ob[0][w][1]);
    } else if constexpr (FP8) {
      dequant_pair8_fp8<DT, UNIT>(word8(st[0], w, 0, 0), word8(st[0], w, 0, 1), word8(st[0], w, 1, 0),
                                  word8(st[0], w, 1, 1), CHANNEL ? 0u : st[0].sc[w], ob[0][w][0], ob[0][w][1]);
    } else {
      dequant_pair8<DT, UNIT>(word8(st[0], w, 0, 0), word8(st[0], w, 0, 1), word8(st[0], w, 1, 0),
                              word8(st[0], w, 1, 1), CHANNEL ? 0u : st[0].sc[w], ob[0][w][0], ob[0][w][1]);
    }
  }
  __syncthreads();

  // One k-step: 64 MFMAs on ob[CUR].  The matrix pipe takes 16 cycles per MFMA, so between every two MFMAs
  // one register of the next k-step's operands (3-5 VALU instructions) is dequantised into ob[CUR ^ 1]; the
  // scheduling barriers keep the compiler from regrouping that into MFMA-only and VALU-only blocks, which would
  // leave the matrix pipe idle during the VALU blocks.
  // The A operands of the next k-step are read from LDS during the last word, each right behind the last MFMA that uses its registers: a whole
  // word of MFMAs covers the reads.  With the chunk's second k-step (CUR) that is the next chunk, which is therefore stored two words, and the
  // workgroup's barrier passed one word, before the end.
  auto a_frags = [&](int buf, int kk) { return (const u32x4*)(lds + buf * (FB_ABUF / 4)) + (kk * FB_MB) * 64 + lane; };
  u32x4 af[FB_MB];
#pragma unroll
  for (int mb = 0; mb < FB_MB; ++mb) af[mb] = a_frags(0, 0)[mb * 64];
  auto kstep = [&](auto cur_tag, int buf, const Stage& nxt, auto refresh_tag) __attribute__((always_inline)) {
    constexpr int CUR = decltype(cur_tag)::value;
    const u32x4* anext = CUR ? a_frags(buf ^ 1, 0) : a_frags(buf, 1);
    if constexpr (CONSTS && decltype(refresh_tag)::value) {
#pragma unroll
      for (int w = 0; w < 4; ++w) ccs[w] = col_const(nxt, w);
    }
    // integer weights: the three dependent stages of one operand register (nibbles -> exact fp16 pair, minus the zero point (bf16: times the scale
    // too, in fp32), times the scale (bf16: the pack)) are spread over three consecutive MFMA pairs, so that no VALU
    // instruction reads the result of the one issued just before it
    uint32_t ph = 0;
    PieceValue<DT> pv;
    auto stage_a = [&](auto p_tag) {  // piece P: nibbles -> (1024+q | 64+q) fp16 pair
      constexpr int P = decltype(p_tag)::value, w = P >> 3, J = P & 7;
      ph = piece_halves<J>((J & 3) < 2 ? nxt.b0[w] : nxt.b1[w]);
    };
    auto stage_b = [&](auto p_tag) {
      constexpr int P = decltype(p_tag)::value, w = P >> 3, J = P & 7;
      pv = piece_value<DT, J>(ph, ccs[w]);
    };
    if constexpr (CONSTS) {
      stage_a(std::integral_constant<int, 0>{});
      stage_b(std::integral_constant<int, 0>{});
      stage_a(std::integral_constant<int, 1>{});
    }
    auto word = [&](auto w_tag) __attribute__((always_inline)) {
      constexpr int w = decltype(w_tag)::value;
      const Fp4Scales fs = fp4_scales(nxt, w);
      uint32_t zs = 0;
      if constexpr (ZPF) zs = as_u32(as_h2(nxt.zf[w]) * as_h2(nxt.sc[w]));
      const uint32_t xa = nxt.b0[w], xb = nxt.b1[w];
      auto step = [&](auto j_tag) __attribute__((always_inline)) {
        constexpr int J = decltype(j_tag)::value;
        mfma_inplace<DT>(acc[J][w][0], af[J], ob[CUR][w][0]);
        mfma_inplace<DT>(acc[J][w][1], af[J], ob[CUR][w][1]);
        uint32_t r;
        if constexpr (w == 3) af[J] = anext[J * 64];
        if constexpr (CONSTS) {
          constexpr int P = 8 * w + J;
          r = piece_finish<DT, UNIT, J>(pv, ccs[w]);
          if constexpr (P + 1 < 32) stage_b(std::integral_constant<int, P + 1>{});
          if constexpr (P + 2 < 32) stage_a(std::integral_constant<int, P + 2>{});
        } else if constexpr (ZPF)
          r = dequant_piece_zpf<J>(xa, xb, nxt.sc[w], zs);
        else if constexpr (FP4 != 0)
          r = ((J & 3) < 2) ? dequant_piece_fp4<DT, J>(xa, fs.a0, fs.a1) : dequant_piece_fp4<DT, J>(xb, fs.b0, fs.b1);
        else
          r = dequant_piece8<DT, UNIT, FP8, J>(word8(nxt, w, (J & 3) >> 1, 0), word8(nxt, w, (J & 3) >> 1, 1),
                                               CHANNEL ? 0u : nxt.sc[w]);
        if constexpr (J < 4)
          ob[CUR ^ 1][w][0][J] = r;
        else
          ob[CUR ^ 1][w][1][J - 4] = r;
        __builtin_amdgcn_sched_barrier(0);
      };
      step(std::integral_constant<int, 0>{});
      step(std::integral_constant<int, 1>{});
      step(std::integral_constant<int, 2>{});
      step(std::integral_constant<int, 3>{});
      step(std::integral_constant<int, 4>{});
      step(std::integral_constant<int, 5>{});
      step(std::integral_constant<int, 6>{});
      step(std::integral_constant<int, 7>{});
    };
    word(std::integral_constant<int, 0>{});
    word(std::integral_constant<int, 1>{});
    if constexpr (CUR) {
      store_a(buf ^ 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    word(std::integral_constant<int, 2>{});
    if constexpr (CUR) {
      __syncthreads();
      __builtin_amdgcn_sched_barrier(0);
    }
    word(std::integral_constant<int, 3>{});
  };
  const std::integral_constant<int, 0> even{};
  const std::integral_constant<int, 1> odd{};

  // ---- main loop: two chunks (four k-steps = the weight ring) per iteration.  The last k-step of an iteration
  // dequantises the first k-step of the next 128 rows of K: the constants are rebuilt there,
  // and in the other three k-steps too when a group is shorter than 128 rows.
  const std::bool_constant<!ONCE && !(CONSTS && CHANNEL)> every{};
#pragma unroll 1
  for (int c0 = 0; c0 < nchunks; c0 += 2) {
    const int ks0 = 2 * c0;
    // chunk c0 in buffer 0
    load_a(c0 + 1);
    kstep(even, 0, st[1], every);
    if constexpr (ONCE) issue_scales(ks0 + 4);
    issue(st[0], ks0 + 4);
    kstep(odd, 0, st[2], every);
    issue(st[1], ks0 + 5);
    // chunk c0+1 in buffer 1
    load_a(c0 + 2);
    kstep(even, 1, st[3], every);
    issue(st[2], ks0 + 6);
    kstep(odd, 1, st[0], std::true_type{});
    issue(st[3], ks0 + 7);
  }

  // ------------------------------------------------------------------------------ epilogue
  // (the inline-asm MFMAs are opaque to the compiler's hazard logic: let the matrix pipe drain before the
  //  accumulators are read)
  asm volatile("s_nop 15\n\ts_nop 15\n\ts_nop 15" ::: "memory");
  // per wavefront and m-block: accumulators -> private LDS slab [16 rows][RED_RS] -> 8-byte row stores
  float* slab = (float*)smem + wv * (16 * RED_RS);
  const int fc4 = (lane & 31) * 4;
  const int fpos = fc4 + (fc4 >= 64 ? 8 : 0);
  const int ncol = cp * 128 + fc4;
  const bool fcol_ok = wave_on && ncol < p.N;
  const bool act = MOE && p.act;
  // cs / bs: channel (and global) scale and bias of the thread's four columns; cu / bu: of the up half's columns
  float cs[4] = {1.f, 1.f, 1.f, 1.f}, bs[4] = {0.f, 0.f, 0.f, 0.f}, cu[4] = {1.f, 1.f, 1.f, 1.f}, bu[4] = {0.f, 0.f, 0.f, 0.f};
  if constexpr (FP4 == 1) {
    // NVFP4 global scale: stored times 2^7 (fp16) / 2^119 (bf16) by the reference's load-time processing
    const uint16_t gv = *(const uint16_t*)p.gscale;
    const float gs = (DT == DT_F16) ? f16_lo_f32(gv) * 0x1.0p-7f : bf16_lo_f32(gv) * 0x1.0p-119f;
#pragma unroll
    for (int j = 0; j < 4; ++j) cs[j] = gs;
  }
  auto col_consts = [&](int col, float* sc_out, float* b_out) {
    const int base = col & ~31, cl = col & 31;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (CHANNEL) {
        const uint16_t sv = Sc[base + single_perm_pos(cl + j)];
        sc_out[j] = ((DT == DT_F16) ? f16_lo_f32(sv) : bf16_lo_f32(sv)) * (FP8 ? fp8_scale_unbias<DT>() : 1.0f);
      }
      if (bias) {
        const uint16_t bv = bias[base + single_perm_pos(cl + j)];
        b_out[j] = (DT == DT_F16) ? f16_lo_f32(bv) : bf16_lo_f32(bv);
      }
    }
  };
  // fused SiLU-and-mul, unsplit: lane -> row (lane >> 4) + 4 i, gate columns 4 (lane & 15) .. + 3 and the up columns of
  // the same outputs, so that all 64 lanes take part
  const int ac4 = (lane & 15) * 4;
  const int ocol = cp * 64 + ac4;
  if (act) {
    if (wave_on) {
      col_consts(ocol, cs, bs);
      col_consts((p.N >> 1) + ocol, cu, bu);
    }
  } else if (fcol_ok) {
    col_consts(ncol, cs, bs);
  }
#pragma unroll
  for (int mb = 0; mb < FB_MB; ++mb) {
#pragma unroll
    for (int w = 0; w < 4; ++w)
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int r = 0; r < 4; ++r) slab[(4 * g + r) * RED_RS + 72 * h + 16 * w + 8 * hf + c] = acc[mb][w][hf][r];
    __builtin_amdgcn_wave_barrier();
    if (act && nsplit == 1) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r16 = (lane >> 4) + 4 * i;
        const int crow = s_crow[mb * 16 + r16];
        if (crow < 0 || !wave_on) continue;
        f32x4 v = *(const f32x4*)(slab + r16 * RED_RS + ac4);
        f32x4 u = *(const f32x4*)(slab + r16 * RED_RS + ac4 + 72);
        const float tw = p.mul_topk ? s_tw[mb * 16 + r16] : 1.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          v[j] = (v[j] * cs[j] + bs[j]) * tw;
          u[j] = (u[j] * cu[j] + bu[j]) * tw;
        }
        store_row4_silu_mul<DT>(p, crow, ocol, v, u);
      }
      __builtin_amdgcn_wave_barrier();
      continue;
    }
    // (a row's read and store in one round waits for each read by itself: 1.006 of the time, 24 dense layers of 669 to 2926 rows, at most 1.019 where K is
    //  short, and 1.008, at most 1.023, both GEMMs of 20 layers with MoE blocks of 128)
    f32x4 rows[8];
    int crows[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r16 = (lane >> 5) + 2 * i;
      crows[i] = MOE ? s_crow[mb * 16 + r16] : row0 + mb * 16 + r16;
      rows[i] = *(const f32x4*)(slab + r16 * RED_RS + fpos);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r16 = (lane >> 5) + 2 * i, crow = crows[i];
      f32x4 v = rows[i];
      if (!fcol_ok || (MOE ? crow < 0 : crow >= p.M)) continue;
      if (MOE && nsplit > 1) {
        // a K piece: the fp32 partial tile [row 128][column 512] goes to scratch; the pass launched behind finishes the rows
        *(f32x4*)(p.ctmp + (((int64_t)part * nsplit + split) * FB_BM + mb * 16 + r16) * 512 + wv * 128 + fc4) = v;
        continue;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = v[j] * cs[j] + bs[j];
      if (MOE && p.mul_topk) {
        const float tw = s_tw[mb * 16 + r16];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] *= tw;
      }
      store_row4<DT, MOE>(p, crow, ncol, v);
    }
    __builtin_amdgcn_wave_barrier();
  }
}

typedef void (*fat_fn)(const KParams);

template <int DT, bool ZP, bool MOE>
static fat_fn pick_fat3(bool channel, bool once) {
  if (channel) return fat_kernel<DT, ZP, true, 4, false, 0, false, MOE, true>;
  return once ? fat_kernel<DT, ZP, false, 4, false, 0, false, MOE, true> : fat_kernel<DT, ZP, false, 4, false, 0, false, MOE, false>;
}
template <int DT, bool MOE>
static fat_fn pick_fat2(bool zp, bool channel, bool once) {
  if (zp) return pick_fat3<DT, true, MOE>(channel, once);
  return pick_fat3<DT, false, MOE>(channel, once);
}
template <int DT>
static fat_fn pick_fat8(bool fp8, bool channel) {
  if (fp8) return channel ? fat_kernel<DT, false, true, 8, true> : fat_kernel<DT, false, false, 8, true>;
  return channel ? fat_kernel<DT, false, true, 8, false> : fat_kernel<DT, false, false, 8, false>;
}

int launch_fat(const w4a16_gemm_args* a, const Plan& pl, hipStream_t stream) {
  const bool zp = a->b_zeros != nullptr, channel = pl.gm == GM_CHANNEL;
  const bool moe = (a->flags & W4A16_F_MOE) != 0, once = pl.group_ksteps >= 4;
  fat_fn fn;
  if (moe) {
    if ((a->flags & W4A16_F_ZP_FLOAT) || (a->wtype != W4A16_WTYPE_U4B8 && a->wtype != W4A16_WTYPE_U4) || pl.dyn_slots <= 0)
      return fail(W4A16_EINVAL, "unsupported kernel variant");
    fn = a->dtype == DT_F16 ? pick_fat2<DT_F16, true>(zp, channel, once) : pick_fat2<DT_BF16, true>(zp, channel, once);
  } else if (a->flags & W4A16_F_ZP_FLOAT) {
    if (a->dtype != DT_F16 || channel) return fail(W4A16_EINVAL, "unsupported kernel variant");
    fn = fat_kernel<DT_F16, false, false, 4, false, 0, true>;
  } else if (a->wtype == W4A16_WTYPE_FE2M1) {
    if (zp || channel) return fail(W4A16_EINVAL, "unsupported kernel variant");
    fn = a->global_scale ? (a->dtype == DT_F16 ? fat_kernel<DT_F16, false, false, 4, false, 1>
                                               : fat_kernel<DT_BF16, false, false, 4, false, 1>)
                         : fat_kernel<DT_BF16, false, false, 4, false, 2>;
  } else if (a->wtype == W4A16_WTYPE_U8B128 || a->wtype == W4A16_WTYPE_FE4M3) {
    const bool fp8 = a->wtype == W4A16_WTYPE_FE4M3;
    if (zp) return fail(W4A16_EINVAL, "unsupported kernel variant");
    fn = a->dtype == DT_F16 ? pick_fat8<DT_F16>(fp8, channel) : pick_fat8<DT_BF16>(fp8, channel);
  } else {
    fn = a->dtype == DT_F16 ? pick_fat2<DT_F16, false>(zp, channel, once) : pick_fat2<DT_BF16, false>(zp, channel, once);
  }
  KParams p = make_kparams(a, pl);
  if (pl.tiles <= 0) return 0;
  // MoE: at most dyn_slots pieces behind the whole tiles (the device knows how many), and the pass that adds them
  const int64_t grid = pl.tiles + (moe ? mid_tail_pieces(pl.tiles, pl.dyn_slots) : 0);
  hipLaunchKernelGGL(fn, dim3((unsigned)grid), dim3(256), FB_SMEM, stream, p);
  W4A16_HIP(hipGetLastError());
  if (moe) return launch_fat_reduce(a, pl, p, stream);
  return 0;
}

}  // namespace w4a16
