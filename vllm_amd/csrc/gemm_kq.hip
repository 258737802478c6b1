// W4A16 GEMM for gfx950 with an in-workgroup K split: C[M,N] = A[M,K] * dequant(Bq)[K,N] (+bias), dense, in three shapes.
// First shape, 64-row tiles: 33..128 rows and wide N, where the 64 x 512 tiles of the 64-row kernel are too few to fill
// the chip (the reference's small-batch thread configurations, csrc/quantization/gptq_marlin/gptq_marlin.cu:120-170).
//
//   workgroup tile 64 rows x 256 columns, 8 wavefronts = 2 column pairs x 4 K-quarters: every wavefront owns
//   64 rows x 128 columns (32 v_mfma_f32_16x16x32 per k-step, 128 fp32 accumulators in AGPRs) over a quarter of the
//   K range, two wavefronts per SIMD.
//   weights      streamed global -> registers per wavefront and dequantised one operand register per MFMA, exactly as
//                in the 64-row kernel (B operand = the reference's half(q - z) * half(s)).
//   activations  each K-quarter stages its own 64 rows x 64 K chunk into LDS in MFMA fragment order (its two
//                wavefronts share it), double buffered; one workgroup barrier per two k-steps.
//   epilogue     the four quarters' partial tiles are added through LDS, one 16-row block at a time.
//   split-K      with fewer tiles than compute units (129..~1000 rows of a narrow layer) K is also cut across
//                workgroups, in splits of whole multiples of 512 K rows: the workgroup writes its 64 x 256 fp32 partial
//                tile (already summed over its quarters) to scratch with plain 128-bit stores and kq_reduce_kernel,
//                launched right behind, adds the splits in order and finishes the rows.  A quarter of the 64 x 512
//                kernel's partial bytes for the same number of wavefronts on the problem.
// Compared with 16-row tiles (which re-read and re-convert the weight strip once per 16 rows) every weight is fetched
// and dequantised once per 64 rows; compared with the 64 x 512 tile there are 2 x 4 times as many independent streams.
// The taller shapes of the same kernel (MB = 5 .. 8, Q = 2: 4 wavefronts, one per SIMD, 80 .. 128 rows x 256 columns, K in halves, up to
// 256 accumulators per lane) serve problems that 128 x 512 tiles of the prefill kernel cut badly: every dequantised operand register feeds
// MB row blocks, and the two K halves are added through LDS instead of through memory.  What bounds such a problem is how its tiles fill the
// rounds of 256 workgroups, so the tile's height and the number of K splits across workgroups (of whole multiples of 256 K rows, the last
// may be shorter) follow from the problem, by the times fitted in gemm.hip; a step of 32 K rows costs 0.25 us at 80 rows, 0.40 at 128.
//   fp16, uint4b8, group 128, weights not cached, before (64- and 128-row tiles, unsplit ones only where they fill 3/4 of a round) and now:
// 4096 x 28672 at 160 rows 71 -> 50 us (80-row tiles), 14336 x 4096 at 300 rows 57 -> 48 (80 rows, four splits) and at 1501 rows 189 -> 161
// (96 rows: 16 x 16 tiles instead of 12 x 16), 4096 x 6144 at 768 rows 60 -> 45, 2048 x 3072 at 1501 rows 43 -> 27.
// They also finish the trailing strips of a prefill launch whose last round would be partly filled (KParams.strip0: first 256-column strip
// of the launch).
//   A third shape (MB = 2 .. 4, Q = 8, one column pair: 32 .. 64 rows x 128 columns, 8 wavefronts, each a K eighth) is the general kernel's
// tile with this kernel's loop.  There a wavefront loads, bounces and converts a k-step and then multiplies: VALU and MFMA add up (203 rows:
// 1280 cycles of a SIMD per k-step of 64 x 128, 544 VALU + 512 MFMA).  Here the operands of the next word are made between the MFMAs,
// activations arrive two k-steps at a time in rows of 128 bytes (17 cycles of the memory pipe per KB; rows of 64 bytes take 34) and are in
// LDS one chunk ahead, scales come and constants are made once per 128 rows of K.  A K part is one wavefront, so nothing in the loop waits
// for another and parts may differ in length.  Accumulators of 32- and 48-row tiles are VGPRs: without AGPRs all 256 registers can hold
// operands.  fp16 uint4b8 / bf16 with zero points, weights not cached, before and now: 4096 x 28672 at 37 rows 24.6 -> 22.5 / 25.1 -> 23.8 us,
// at 64 rows 29.5 -> 25.9 / 31.2 -> 28.7; 4096 x 6144 at 203 rows 23.6 -> 19.5 / 26.1 -> 21.1; 4096 x 4096 at 300 rows 23.0 -> 18.7 / 25.8 -> 20.7.
// (The weights of 4096 x 28672 in the 256 MB cache: at 64 rows 29.1 -> 23.2 / 31.5 -> 28.2.)
// Groups of 32 and 64 rows have a variant with scales in every k-step's stage and constants made for every word (SHORT; a k-step costs it
// 1 % more in fp16, 9 % in bf16, 16 % with zero points; 64-row tiles with zero points would spill 2 to 18 registers and do not exist): of
// 660 problems of 17 to 512 rows with such groups it takes 162, to 0.87 of their time in the mean, worst 1.01.
// Requirements (host-checked): K % 512 == 0 (taller shapes: K % 256 == 0, third shape: K % 128 == 0), so that every K part runs whole ring
// periods of 4 k-steps; scales grouped (a power-of-two number of k-steps) or channelwise, no per-row g_idx, A's columns already in
// weight order.
#include <type_traits>

#include "gemm_kernels.h"

namespace w4a16 {

constexpr int KQ_D = 4;      // weight k-steps in flight per wavefront
// MB m-blocks of 16 rows per tile, K cut into Q parts inside the workgroup (2 Q wavefronts)
// dwords of one k-step of an A buffer: MB m-blocks x 64 lanes x 16 B, and half a row of the 64 banks: a wavefront's staging stores, 8 rows x
// 2 k-steps x 4 dwords, then hit 64 different ones (128-row tiles without: 4096 x 4096 at 1024 rows 41.4 us, 41.6 with, and three spills)
constexpr int kq_kstep(int MB) { return MB * 256 + (MB < 8 ? 32 : 0); }
constexpr int kq_abuf(int MB) { return 2 * kq_kstep(MB) * 4; }  // one A buffer of one K part: 2 k-steps
constexpr int KQ_RS = 76;  // floats per row of an epilogue slab of 64 columns (40 for the half of either n-tile: conflict-free, 16-byte aligned)
constexpr int kq_smem(int MB, int Q, int WN) {
  // staging rings | what the parts hand each other in the epilogue.  64 x 256 and 32 x 128 tiles 74 KB, 48 and 64 x 128 100 and 132, tall ones 80 to 128:
  // one workgroup to a compute unit, which is what their registers leave room for.  (Four and eight parts with two m-blocks at a time, 148 KB: level, 1.001
  // of the time in the mean of 90 problems of 80 to 967 rows, weights not cached, none beyond 1.012 either way.)
  const int stage = Q * 2 * kq_abuf(MB), boxes = Q == 2 ? WN * Q * MB * 4096 : WN * Q * 16 * RED_RS * 4;
  return stage > boxes ? stage : boxes;
}

// channel scale and bias of four finished columns starting at `ncol` (scales and bias are stored permuted); 1 and 0 are the caller's
template <int DT, bool CHANNEL>
__device__ __forceinline__ void kq_col_consts(const KParams& p, int ncol, float* cs, float* bs) {
  const uint16_t *Sc = (const uint16_t*)p.S, *bias = (const uint16_t*)p.bias;
  const int base = ncol & ~31, cl = ncol & 31;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (CHANNEL) cs[j] = lo_f32<DT>(Sc[base + single_perm_pos(cl + j)]);
    if (bias) bs[j] = lo_f32<DT>(bias[base + single_perm_pos(cl + j)]);
  }
}

// SHORT: private parts and tall tiles with groups below 128 rows, whose scales and constants come with every k-step.  (Tall tiles had both loops in
// one kernel, 40 to 80 registers more, and scales in every k-step for every group: 80 to 112 rows, groups of 32 and 64 0.90 - 0.97 of the
// time, of 128 0.96 - 1.00, reading A early included; 14336 x 4096 at 1501 rows, fp16, groups of 128: 166 -> 160 us.)
template <int DT, bool ZP, bool CHANNEL, int MB = 4, int Q = 4, int WN = 2, bool SHORT = false>
__global__ __launch_bounds__(64 * WN * Q) void kq_kernel(const KParams p) {
  static_assert((MB == 4 && Q == 4 && WN == 2) || (MB > 4 && MB <= 8 && Q == 2 && WN == 2) || (MB >= 2 && MB <= 4 && Q == 8 && WN == 1),
                "64 x 256 in K quarters, 80 .. 128 x 256 in K halves or 32 .. 64 x 128 in K eighths");
  constexpr int KQ_MB = MB, KQ_BM = 16 * MB, KQ_Q = Q, KQ_ABUF = kq_abuf(MB), KQ_TN = 128 * WN;
  constexpr bool PRIV = (WN == 1);  // a K part is one wavefront: it stages its own activations, nothing in the loop waits for another
  // HOIST: the dequantisation constants of the four word positions are kept for the k-step whose operands are being built.  A loop
  // iteration covers four k-steps (128 rows of K, aligned: every K part starts at a multiple of four k-steps), so with groups of
  // 128 rows or more, or one scale per column, they are rebuilt once per iteration instead of once per k-step.  (Not where the registers
  // are short: 64-row tiles keep them in the 128-column form only, and there not in bf16 with grouped scales: 12 to 28 would spill.)
  constexpr bool ONCE = !SHORT && (PRIV || KQ_MB > 4);
  constexpr bool HOIST = KQ_MB > 4 || (PRIV && ONCE && (KQ_MB < 4 || CHANNEL || DT == DT_F16));
  // EARLY: the A operands of the next k-step are read from LDS during this one's last word, and the next chunk is stored and the barrier passed
  // before that; 80 to 112 rows then load chunks two ahead, being stored half a k-step sooner.  Time over reading at the start of the k-step:
  // 64 x 256 0.99, 80 to 112 rows 0.98 (fp16 uint4b8 0.97, channel-wise 0.99); 128 rows, whose words are longer, 1.015, private parts, which have
  // two wavefronts to a SIMD and no barrier, 1.00 - 1.02: these two don't.
  constexpr bool EARLY = !PRIV && KQ_MB < 8;
  constexpr bool UNIT = CHANNEL;
  extern __shared__ __align__(16) unsigned char smem[];
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wn = wv % WN, q = wv / WN;  // column pair inside the tile, K part
  const int c = lane & 7, h = (lane >> 3) & 1, g = lane >> 4;

  // tile order: consecutive workgroups walk M first, so workgroups resident together share weight strips
  const int mtiles = (p.M + KQ_BM - 1) / KQ_BM;
  // (workgroup ids rotate over the eight XCDs; with xcd_map each takes a contiguous run of the tiles, and its L2 a share of the strips)
  const int xcd = blockIdx.x & 7, rem = gridDim.x & 7;
  const int wg = p.xcd_map ? xcd * (int)(gridDim.x >> 3) + min(xcd, rem) + (int)(blockIdx.x >> 3) : (int)blockIdx.x;
  const int mt = wg % mtiles;
  const int split = (wg / mtiles) % p.splits, strip = wg / (mtiles * p.splits);
  const int cp = (p.strip0 + strip) * WN + wn;  // column pair of this wavefront (strip0: first 256-column strip of the launch)
  const bool wave_on = cp * 128 < p.N;          // N not a multiple of 256: the trailing wavefronts only help staging
  const int row0 = mt * KQ_BM;

  const uint32_t* Bq = p.B;
  const uint16_t* Sc = (const uint16_t*)p.S;
  const uint32_t* Zp = p.Z;
  // ---- weights of this wavefront
  const int nt = (wave_on && (2 * cp + h) * 64 < p.N) ? 2 * cp + h : 0;
  const int64_t b_row = p.N >> 1;
  const u32x4* bp = (const u32x4*)Bq + nt * 32 + (4 * c + g);
  const int64_t s_row = p.N >> 3;
  const u32x4* sp = (const u32x4*)Sc + nt * 8 + c;
  const uint32_t* zp = ZP ? Zp + nt * 8 + c : nullptr;

  // ---- this quarter's k-steps: [ks_b, ks_e), a multiple of 4 long
  // (host: whole splits and the rest behind them are multiples of 4 Q k-steps, so the parts of a workgroup are equally long)
  // (private parts: as equally long as multiples of 4 k-steps go, some may be empty)
  const int in_split = min(p.ksteps_per_split, p.total_ksteps - split * p.ksteps_per_split);
  const int ks_b = split * p.ksteps_per_split + (PRIV ? in_split / 4 * q / KQ_Q * 4 : q * (in_split / KQ_Q));
  const int per_q = PRIV ? in_split / 4 * (q + 1) / KQ_Q * 4 - in_split / 4 * q / KQ_Q * 4 : in_split / KQ_Q, ks_e = ks_b + per_q;

  // ---- activation staging: the K part's 128 threads; thread tq loads piece (tq & 7) of tile rows (tq >> 3) + 16 i
  // (rows without a source read row 0 of A; their results are never stored)
  // (private parts: its 64 threads, rows (tq >> 3) + 8 i, MB / NH of them at a time, the last row of the problem in place of the rows
  //  behind it)
  constexpr int AR = PRIV ? 8 : 16, AN = KQ_BM / AR;           // rows per load instruction, loads per chunk
  constexpr int NH = PRIV && KQ_MB == 4 ? 2 : 1, AH = AN / NH;  // (64 rows: the chunk in two halves, for its registers)
  constexpr int AD = EARLY && KQ_MB > 4 ? 2 : 1;                // chunks in flight
  const int tq = wn * 64 + lane;
  const int piece = tq & 7;
  const uint16_t* arow[PRIV ? 1 : AN];
  uint32_t aoff[PRIV ? AN : 1];
  const char* abase = (const char*)p.A + (int64_t)row0 * p.lda * 2;
#pragma unroll
  for (int i = 0; i < AN; ++i) {
    if constexpr (PRIV) {
      aoff[i] = (uint32_t)min((tq >> 3) + AR * i, p.M - 1 - row0) * ((uint32_t)p.lda * 2) + piece * 16;  // (the host checks the size)
    } else {
      const int src = row0 + (tq >> 3) + AR * i;
      arow[i] = (const uint16_t*)p.A + (int64_t)(src < p.M ? src : 0) * p.lda + piece * 8;
    }
  }
  // LDS A layout per part: [buffer][k-step 2][m-block][lane 64][4 dwords]; the 16 bytes of (row, piece) are the
  // K pairs 8*pp + 2j (pp = piece & 3), which belong to lane (j*16 + row%16), dword pp, of k-step piece >> 2.
  uint32_t* lds = (uint32_t*)smem + q * (2 * KQ_ABUF / 4);
  const int a_wr0 = (piece >> 2) * kq_kstep(KQ_MB) + (tq >> 3) * 4 + (piece & 3);
  u32x4 areg[AD][AH];
  // (chunk and k-step indices are clamped instead of guarded: the last iteration re-reads its own data, which
  //  keeps the main loop free of branches)
  auto load_a = [&](int chunk, int half, int slot = 0) {  // chunk: relative to ks_b
    chunk = min(ks_b / 2 + chunk, ks_e / 2 - 1);
#pragma unroll
    for (int i = 0; i < AH; ++i) {
      if constexpr (PRIV)
        areg[slot][i] = *(const u32x4*)(abase + (int64_t)chunk * 128 + aoff[half * AH + i]);
      else
        areg[slot][i] = *(const u32x4*)(arow[i] + chunk * 64);
    }
  };
  auto store_a = [&](int buf, int half, int slot = 0) {
    uint32_t* dst = lds + buf * (KQ_ABUF / 4) + a_wr0;
#pragma unroll
    for (int i = 0; i < AH; ++i) {
      const int r = AR * (half * AH + i);  // (row (tq >> 3) + r: m-block r / 16, AR = 8: upper half of it for odd loads)
#pragma unroll
      for (int j = 0; j < 4; ++j) dst[(r / 16) * 256 + (r % 16) * 4 + j * 64] = areg[slot][i][j];
    }
  };
  // (a wavefront's LDS accesses are executed in order; that they stay in this order is for the compiler to know)
  auto loop_barrier = [&]() {
    if constexpr (PRIV) {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
      __builtin_amdgcn_wave_barrier();
    } else {
      __syncthreads();
    }
  };

  struct Stage {
    u32x4 b0, b1, sc;
    uint32_t zq;
  };
  Stage st[KQ_D];
  // groups of 128 rows at least (host): scales and zero points once per loop iteration, loaded with its first k-step
  u32x4 sc128 = {0, 0, 0, 0}, sc_now = {0, 0, 0, 0};
  uint32_t zq128 = 0, zq_now = 0;
  auto next_scales = [&]() { sc_now = sc128, zq_now = zq128; };
  auto issue_scales = [&](int ks) {
    const int gi = CHANNEL ? 0 : min(ks_b + ks, ks_e - 1) >> p.group_shift;
    if (!CHANNEL) sc128 = sp[(int64_t)gi * s_row];
    if (ZP) zq128 = zp[(int64_t)gi * s_row];
  };
  auto issue = [&](Stage& s, int ks) {  // ks: relative to ks_b
    ks = min(ks_b + ks, ks_e - 1);
    int gi = 0;
    if (!CHANNEL) gi = ks >> p.group_shift;
    if (!CHANNEL && !ONCE) s.sc = sp[(int64_t)gi * s_row];
    if (ZP && !ONCE) s.zq = zp[(int64_t)gi * s_row];
    s.b0 = bp[(int64_t)(2 * ks) * b_row];
    s.b1 = bp[(int64_t)(2 * ks + 1) * b_row];
  };
  auto col_const = [&](const Stage& s, int w) {
    return make_col_const<DT, UNIT>(CHANNEL ? 0u : ONCE ? sc_now[w] : s.sc[w], ZP ? zero_pair(ONCE ? zq_now : s.zq, w) : ZERO_U4B8);
  };

  f32x4 acc[KQ_MB][4][2];
#pragma unroll
  for (int mb = 0; mb < KQ_MB; ++mb)
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      acc[mb][w][0] = f32x4{0, 0, 0, 0};
      acc[mb][w][1] = f32x4{0, 0, 0, 0};
    }

  const int nchunks = per_q / 2;  // even

  // ---- prologue
  const bool any = !PRIV || nchunks > 0;
  if (any) {
#pragma unroll
    for (int hf = 0; hf < NH; ++hf) {
      load_a(0, hf);
      if constexpr (AD == 2) load_a(1, 0, 1);
      if (hf == 0) {
        if constexpr (ONCE) issue_scales(0);
#pragma unroll
        for (int j = 0; j < KQ_D; ++j) issue(st[j], j);
      }
      store_a(0, hf);
    }
  }
  // B operands of two Marlin words: the one whose MFMAs are being issued and the one being dequantised
  u32x4 ob[2][2];
  ColConst<DT> ccs[4];
  if (any) {
    next_scales();
#pragma unroll
    for (int w = 0; w < 4; ++w) ccs[w] = col_const(st[0], w);
    dequant_pair<DT, UNIT>(st[0].b0[0], st[0].b1[0], ccs[0], ob[0][0], ob[0][1]);
  }
  __syncthreads();

  // One k-step: per Marlin word w, 2 MB MFMAs on ob[w & 1]; after each MFMA (MB = 8: pair of MFMAs) one register of the following word's
  // operands (word w + 1 of this k-step, or word 0 of the next k-step `nxt`) is finished into ob[(w + 1) & 1].  A register is made in three
  // dependent steps; behind an MFMA stand the last of one register, the second of the next and the first of the one after that, none of
  // which waits for another (in one chain: 12 % of the loop at six such instructions per MFMA and two wavefronts per SIMD).
  // The scheduling barriers keep the compiler from regrouping this into MFMA-only and VALU-only blocks.
  // (EARLY: each operand right behind the last MFMA that uses its registers)
  auto a_frags = [&](int buf, int kk) { return (const u32x4*)(lds + buf * (KQ_ABUF / 4) + kk * kq_kstep(KQ_MB)) + lane; };
  u32x4 af[KQ_MB];
  if constexpr (EARLY) {
#pragma unroll
    for (int mb = 0; mb < KQ_MB; ++mb) af[mb] = a_frags(0, 0)[mb * 64];
  }
  auto kstep = [&](int buf, auto kk_tag, const Stage& cur, const Stage& nxt, auto refresh_tag) __attribute__((always_inline)) {
    constexpr bool REFRESH = decltype(refresh_tag)::value, KK = decltype(kk_tag)::value;
    const u32x4* anext = KK ? a_frags(buf ^ 1, 0) : a_frags(buf, 1);
    if constexpr (!EARLY) {
#pragma unroll
      for (int mb = 0; mb < KQ_MB; ++mb) af[mb] = a_frags(buf, KK)[mb * 64];
    }
    ColConst<DT> ccw[2];  // !HOIST: of the word being made and of the one behind it
    if constexpr (!HOIST) {
      if constexpr (ONCE) asm volatile("" : "+v"(sc_now), "+v"(zq_now));  // (or the compiler keeps all four words' constants)
      ccw[0] = col_const(cur, 1);
    }
    // register P of the k-step: J = P & 7 of the word behind word P >> 3
    auto consts = [&](auto p_tag) -> const ColConst<DT>& {
      constexpr int W = decltype(p_tag)::value >> 3;
      return HOIST ? ccs[(W + 1) & 3] : ccw[W & 1];
    };
    uint32_t halves = 0;
    PieceValue<DT> value;
    auto make_halves = [&](auto p_tag) {
      constexpr int P = decltype(p_tag)::value, W = P >> 3, J = P & 7;
      const Stage& src = W == 3 ? nxt : cur;
      halves = piece_halves<J>((J & 3) < 2 ? src.b0[(W + 1) & 3] : src.b1[(W + 1) & 3]);
    };
    make_halves(std::integral_constant<int, 0>{});
    value = piece_value<DT, 0>(halves, consts(std::integral_constant<int, 0>{}));
    make_halves(std::integral_constant<int, 1>{});
    auto step = [&](auto p_tag) __attribute__((always_inline)) {
      constexpr int P = decltype(p_tag)::value, w = P >> 3, J = P & 7, wn2 = (w + 1) & 3;
      if constexpr (EARLY && KK && P == 16) store_a(buf ^ 1, NH - 1, buf ? 0 : AD - 1);
      if constexpr (EARLY && KK && P == 24) loop_barrier();
#pragma unroll
      for (int i = J * KQ_MB / 4; i < (J + 1) * KQ_MB / 4; ++i) {
        if constexpr (KQ_MB < 4)
          mfma_inplace_v<DT>(acc[i >> 1][w][i & 1], af[i >> 1], ob[w & 1][i & 1]);
        else
          mfma_inplace<DT>(acc[i >> 1][w][i & 1], af[i >> 1], ob[w & 1][i & 1]);
        if constexpr (EARLY && w == 3)
          if (i & 1) af[i >> 1] = anext[(i >> 1) * 64];
      }
      ob[wn2 & 1][J >> 2][J & 3] = piece_finish<DT, UNIT, J>(value, consts(p_tag));
      // the constants the next registers want: of `nxt` where the k-step ends a group, each as soon as the old ones have been used
      if constexpr (w == 2 && J == 4 && ONCE && REFRESH) next_scales();
      if constexpr (HOIST) {
        if constexpr (REFRESH && w == 2 && J == 4) ccs[0] = col_const(nxt, 0);
        if constexpr (REFRESH && w == 3 && J == 1) ccs[1] = col_const(nxt, 1);
        if constexpr (REFRESH && w == 3 && J == 3) ccs[2] = col_const(nxt, 2);
        if constexpr (REFRESH && w == 3 && J == 5) ccs[3] = col_const(nxt, 3);
      } else if constexpr (w < 3 && J == 4) {
        if constexpr (ONCE) asm volatile("" : "+v"(sc_now), "+v"(zq_now));
        ccw[wn2 & 1] = col_const(w == 2 ? nxt : cur, (w + 2) & 3);
      }
      if constexpr (P + 1 < 32) value = piece_value<DT, (P + 1) & 7>(halves, consts(std::integral_constant<int, P + 1>{}));
      if constexpr (P + 2 < 32) make_halves(std::integral_constant<int, P + 2>{});
      __builtin_amdgcn_sched_barrier(0);
    };
    for_each_piece<32>(step);
  };
  auto end_chunk = [&](int buf) {
    if constexpr (!EARLY) {
      store_a(buf ^ 1, NH - 1);
      loop_barrier();
    }
  };

  // ---- main loop: two chunks (four k-steps = the weight ring) per iteration; the K parts of a workgroup run the same count,
  // but private ones, which may have one iteration more or fewer, or none.  The
  // last k-step of an iteration builds the first operands of the next 128 rows of K: the constants are rebuilt there,
  // and in the other three k-steps too when a group is shorter than 128 rows.
  const std::bool_constant<HOIST && !ONCE> every{};
  const std::true_type refresh{};
  Pace pace;
  if constexpr (PRIV) pace.start(nchunks);
#pragma unroll 1
  for (int c0 = 0; c0 < nchunks; c0 += 2) {
    const int ks0 = 2 * c0;
    if constexpr (PRIV) pace.round(c0);
    load_a(c0 + AD, 0);
    kstep(0, std::false_type{}, st[0], st[1], every);
    if constexpr (ONCE) issue_scales(ks0 + 4);
    issue(st[0], ks0 + 4);
    if constexpr (NH == 2) store_a(1, 0), load_a(c0 + 1, 1);
    kstep(0, std::true_type{}, st[1], st[2], every);
    issue(st[1], ks0 + 5);
    end_chunk(0);
    load_a(c0 + AD + 1, 0, AD - 1);
    kstep(1, std::false_type{}, st[2], st[3], every);
    issue(st[2], ks0 + 6);
    if constexpr (NH == 2) store_a(0, 0), load_a(c0 + 2, 1);
    kstep(1, std::true_type{}, st[3], st[0], refresh);
    issue(st[3], ks0 + 7);
    end_chunk(1);
  }

  // ------------------------------------------------------------------------------ epilogue
  // (the inline-asm MFMAs are opaque to the compiler's hazard logic: let the matrix pipe drain before the
  //  accumulators are read)
  asm volatile("s_nop 15\n\ts_nop 15\n\ts_nop 15" ::: "memory");
  // (the last barrier of the loop, or this one, separates what follows from the A buffers it overlays)
  if constexpr (PRIV) __syncthreads();
  const int ncol0 = cp * 128;
  float cs[4] = {1.f, 1.f, 1.f, 1.f}, bs[4] = {0.f, 0.f, 0.f, 0.f};
  int el = t;  // (taken apart again here: a lane's place kept through the loop would spill in one of the kernels)
  asm volatile("" : "+v"(el));
  if constexpr (KQ_Q == 2) {
    // Two parts: each hands the other the fragments (m-block, word, column half: 16 rows x 16 columns, four rows to a lane) of two words of the
    // four and finishes those of the other two, all in one exchange of half the accumulators.  From the loop to the end, 80 rows, four splits: 2.1 us,
    // 3.7 with every m-block through slabs of both parts and two barriers; 96 rows, unsplit 2.9 and 4.9.  14336 x 4096 at 300 rows, fp16, act-order 51.6 ->
    // 50.6 us, 4096 x 6144 at 1501 rows 90.7 -> 87.7.
    float* const boxes = (float*)smem;
    constexpr int BOX = KQ_MB * 4 * 256;  // floats of a wavefront's box: what it gets
    float* const to = boxes + (wv ^ WN) * BOX + (el & 63) * 4;
    float* const box = boxes + wv * BOX;
    auto word_of = [&](int part, int i) { return 2 * part + (i >> 1); };  // fragment i of an m-block: word, half i & 1
    const int lc = (el & 15) * 4, lh = lc >> 5, lpos = lh * 40 + (lc & 31);  // 64 columns: 32 of either n-tile
    const int ncol = ncol0 + 64 * lh + 32 * q + (lc & 31);
    const bool col_ok = wave_on && ncol < p.N;
    if (col_ok && p.splits == 1) kq_col_consts<DT, CHANNEL>(p, ncol, cs, bs);
    auto exchange = [&](auto part_tag) __attribute__((always_inline)) {  // (the part as a constant: accumulators are registers)
      constexpr int PART = decltype(part_tag)::value;
#pragma unroll
      for (int mb = 0; mb < KQ_MB; ++mb)
#pragma unroll
        for (int i = 0; i < 4; ++i) *(f32x4*)(to + (mb * 4 + i) * 256) = acc[mb][word_of(1 - PART, i)][i & 1];
      __syncthreads();
      float* const part_out = p.ctmp + ((((int64_t)(strip * mtiles + mt) * p.splits + split) * WN + wn) * 2 + PART) * (KQ_MB * 1024) + (el & 63) * 4;
      float* const slab = box;  // [2][16 rows][KQ_RS], over what has been read
      constexpr int SLAB = 16 * KQ_RS;
      f32x4 v[KQ_MB][4];
#pragma unroll
      for (int mb = 0; mb < KQ_MB; ++mb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const f32x4 got = *(const f32x4*)(box + (mb * 4 + i) * 256 + (el & 63) * 4), own = acc[mb][word_of(PART, i)][i & 1];
          v[mb][i] = own + got;
        }
      if (p.splits > 1) {
#pragma unroll
        for (int mb = 0; mb < KQ_MB; ++mb)
#pragma unroll
          for (int i = 0; i < 4; ++i) *(f32x4*)(part_out + (mb * 4 + i) * 256) = v[mb][i];
        return;
      }
      __builtin_amdgcn_wave_barrier();
      const int at = 4 * (el >> 4 & 3) * KQ_RS + 40 * (el >> 3 & 1) + (el & 7);
#pragma unroll
      for (int m0 = 0; m0 < KQ_MB; m0 += 2) {
#pragma unroll
        for (int e = 0; e < 2 && m0 + e < KQ_MB; ++e)
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) slab[e * SLAB + at + r * KQ_RS + 8 * i] = v[m0 + e][i][r];
        __builtin_amdgcn_wave_barrier();
        f32x4 rows[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (i < 4 || m0 + 1 < KQ_MB) rows[i] = *(const f32x4*)(slab + (i >> 2) * SLAB + ((el >> 4 & 3) + 4 * (i & 3)) * KQ_RS + lpos);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int crow = row0 + 16 * m0 + (el >> 4 & 3) + 4 * i;
          if ((i < 4 || m0 + 1 < KQ_MB) && col_ok && crow < p.M) {
#pragma unroll
            for (int j = 0; j < 4; ++j) rows[i][j] = rows[i][j] * cs[j] + bs[j];
            store_row4<DT, false>(p, crow, ncol, rows[i]);
          }
        }
        __builtin_amdgcn_wave_barrier();
      }
    };
    if (q == 0)
      exchange(std::integral_constant<int, 0>{});
    else
      exchange(std::integral_constant<int, 1>{});
  } else {
    // per m-block: every wavefront writes its 16 x 128 partial to its slab [16 rows][RED_RS]; after a barrier the wavefront of
    // K part q adds the Q parts' slabs of its column pair for rows (16 / Q) q .. and finishes them.
    float* slabs = (float*)smem;
    const int slab_at = wv * (16 * RED_RS) + 4 * (el >> 4 & 3) * RED_RS + 72 * (el >> 3 & 1) + (el & 7);
    const int fc4 = (lane & 31) * 4;
    const int fpos = fc4 + (fc4 >= 64 ? 8 : 0);
    const int ncol = ncol0 + fc4;
    const bool fcol_ok = wave_on && ncol < p.N;
    if (fcol_ok) kq_col_consts<DT, CHANNEL>(p, ncol, cs, bs);
#pragma unroll
    for (int mb = 0; mb < KQ_MB; ++mb) {
      if (mb > 0) __syncthreads();
#pragma unroll
      for (int w = 0; w < 4; ++w)
#pragma unroll
        for (int hf = 0; hf < 2; ++hf)
#pragma unroll
          for (int r = 0; r < 4; ++r) slabs[slab_at + r * RED_RS + 16 * w + 8 * hf] = acc[mb][w][hf][r];
      __syncthreads();
#pragma unroll
      for (int i = 0; i < 8 / KQ_Q; ++i) {
        const int r16 = (16 / KQ_Q) * q + (lane >> 5) + 2 * i;
        const int crow = row0 + mb * 16 + r16;
        f32x4 v = {0, 0, 0, 0};
#pragma unroll
        for (int qq = 0; qq < KQ_Q; ++qq) v += *(const f32x4*)(slabs + (qq * WN + wn) * (16 * RED_RS) + r16 * RED_RS + fpos);
        if (p.splits > 1) {
          if (crow < p.M)
            *(f32x4*)(p.ctmp + (((int64_t)(strip * mtiles + mt) * p.splits + split) * KQ_BM + mb * 16 + r16) * KQ_TN + wn * 128 + fc4) = v;
        } else if (fcol_ok && crow < p.M) {
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] = v[j] * cs[j] + bs[j];
          store_row4<DT, false>(p, crow, ncol, v);
        }
      }
    }
  }
}

// Second pass of a split-K launch: adds the splits' partial tiles in split order, then channel scale, bias and
// conversion as kq_kernel's own epilogue.  One workgroup per (tile, 16-row block); thread -> 4 columns of 4 rows.
template <int DT, bool CHANNEL, int KQ_TN>
__global__ __launch_bounds__(256) void kq_reduce_kernel(const KParams p, int mb) {
  const int KQ_BM = 16 * mb;
  const int t = threadIdx.x;
  const int mtiles = (p.M + KQ_BM - 1) / KQ_BM;
  const int tile = blockIdx.x / mb, rb = blockIdx.x % mb;
  const int mt = tile % mtiles, strip = tile / mtiles;
  constexpr int TR = 1024 / KQ_TN;  // rows per pass
  const int fc4 = (t % (KQ_TN / 4)) * 4;
  const int ncol = (p.strip0 + strip) * KQ_TN + fc4;
  if (ncol >= p.N) return;
  float cs[4] = {1.f, 1.f, 1.f, 1.f}, bs[4] = {0.f, 0.f, 0.f, 0.f};
  kq_col_consts<DT, CHANNEL>(p, ncol, cs, bs);
  const float* parts = p.ctmp + (int64_t)tile * p.splits * (KQ_BM * KQ_TN) + fc4;
#pragma unroll
  for (int i = 0; i < 16 / TR; ++i) {
    const int r = rb * 16 + t / (KQ_TN / 4) + TR * i;
    const int crow = mt * KQ_BM + r;
    if (crow >= p.M) continue;
    f32x4 v = {0, 0, 0, 0};
    for (int s0 = 0; s0 < p.splits; s0 += 4) {  // (four splits' loads are in flight together)
      f32x4 a[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) a[j] = *(const f32x4*)(parts + ((int64_t)min(s0 + j, p.splits - 1) * KQ_BM + r) * KQ_TN);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (s0 + j < p.splits) v += a[j];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = v[j] * cs[j] + bs[j];
    u32x2 o;
    if constexpr (DT == DT_F16)
      o = u32x2{pack_f16(v[0], v[1]), pack_f16(v[2], v[3])};
    else
      o = u32x2{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
    *(u32x2*)((uint16_t*)p.C + (int64_t)crow * p.N + ncol) = o;
  }
}

// The same behind tall tiles, whose partial tiles are fragments in the order in which their wavefronts hold them: [column pair][K part][m-block]
// [word of two, column half][lane][row of four].  One workgroup per (tile, m-block), a wavefront for each column pair and part.
template <int DT, bool CHANNEL>
__global__ __launch_bounds__(256) void kq_reduce_tall_kernel(const KParams p, int mb) {
  __shared__ __align__(16) float slabs[4][16 * KQ_RS];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;  // wv: 2 wn + part
  const int mtiles = (p.M + 16 * mb - 1) / (16 * mb);
  const int tile = blockIdx.x / mb, m = blockIdx.x % mb;
  const int mt = tile % mtiles, cp = (p.strip0 + tile / mtiles) * 2 + (wv >> 1);
  const int lc = (lane & 15) * 4, lh = lc >> 5;
  const int ncol = cp * 128 + 64 * lh + 32 * (wv & 1) + (lc & 31), row0 = (mt * mb + m) * 16 + (lane >> 4);
  if (row0 - (lane >> 4) >= p.M || cp * 128 >= p.N) return;
  const bool col_ok = ncol < p.N;
  float cs[4] = {1.f, 1.f, 1.f, 1.f}, bs[4] = {0.f, 0.f, 0.f, 0.f};
  if (col_ok) kq_col_consts<DT, CHANNEL>(p, ncol, cs, bs);
  const int64_t piece = mb * 4096;  // floats of a partial tile
  const float* parts = p.ctmp + (int64_t)tile * p.splits * piece + (wv * mb + m) * 1024 + lane * 4;
  f32x4 v[4] = {};
  for (int s0 = 0; s0 < p.splits; s0 += 4) {  // (four splits' loads are in flight together)
    f32x4 a[4][4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) a[j][i] = *(const f32x4*)(parts + min(s0 + j, p.splits - 1) * piece + i * 256);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (s0 + j < p.splits) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] += a[j][i];
      }
  }
  float* slab = slabs[wv];
  const int at = 4 * (lane >> 4) * KQ_RS + 40 * (lane >> 3 & 1) + (lane & 7);
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) slab[at + r * KQ_RS + 8 * i] = v[i][r];
  __builtin_amdgcn_wave_barrier();
  f32x4 rows[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) rows[i] = *(const f32x4*)(slab + ((lane >> 4) + 4 * i) * KQ_RS + lh * 40 + (lc & 31));
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (!col_ok || row0 + 4 * i >= p.M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) rows[i][j] = rows[i][j] * cs[j] + bs[j];
    store_row4<DT, false>(p, row0 + 4 * i, ncol, rows[i]);
  }
}

typedef void (*kq_fn)(const KParams);
typedef void (*kq_reduce_fn)(const KParams, int);

template <int DT, int MB, int Q, int WN>
static kq_fn pick_kq(bool zp, bool channel) {
  if (zp) return channel ? kq_kernel<DT, true, true, MB, Q, WN> : kq_kernel<DT, true, false, MB, Q, WN>;
  return channel ? kq_kernel<DT, false, true, MB, Q, WN> : kq_kernel<DT, false, false, MB, Q, WN>;
}
template <int DT, int MB>
static kq_fn pick_kq_tall(bool zp, bool channel, bool short_groups) {
  if (short_groups) return zp ? kq_kernel<DT, true, false, MB, 2, 2, true> : kq_kernel<DT, false, false, MB, 2, 2, true>;
  return pick_kq<DT, MB, 2, 2>(zp, channel);
}
// (64-row tiles with zero points would spill)
template <int DT, int MB>
static kq_fn pick_kq_short(bool zp) {
  if (!zp) return kq_kernel<DT, false, false, MB, 8, 1, true>;
  if constexpr (MB == 4)
    return nullptr;
  else
    return kq_kernel<DT, true, false, MB, 8, 1, true>;
}
template <int DT>
static kq_fn pick_kq(int mb, int tn, bool zp, bool channel, bool short_groups) {
  if (tn == 128 && short_groups) return mb == 2 ? pick_kq_short<DT, 2>(zp) : mb == 3 ? pick_kq_short<DT, 3>(zp) : mb == 4 ? pick_kq_short<DT, 4>(zp) : nullptr;
  switch (tn == 128 ? -mb : mb) {
    case -2: return pick_kq<DT, 2, 8, 1>(zp, channel);
    case -3: return pick_kq<DT, 3, 8, 1>(zp, channel);
    case -4: return pick_kq<DT, 4, 8, 1>(zp, channel);
    case 4: return pick_kq<DT, 4, 4, 2>(zp, channel);
    case 5: return pick_kq_tall<DT, 5>(zp, channel, short_groups);
    case 6: return pick_kq_tall<DT, 6>(zp, channel, short_groups);
    case 7: return pick_kq_tall<DT, 7>(zp, channel, short_groups);
    case 8: return pick_kq_tall<DT, 8>(zp, channel, short_groups);
    default: return nullptr;
  }
}
template <int DT>
static kq_reduce_fn pick_kq_reduce(int tn, int mb, bool channel) {
  if (mb > 4) return channel ? kq_reduce_tall_kernel<DT, true> : kq_reduce_tall_kernel<DT, false>;
  if (tn == 128) return channel ? kq_reduce_kernel<DT, true, 128> : kq_reduce_kernel<DT, false, 128>;
  return channel ? kq_reduce_kernel<DT, true, 256> : kq_reduce_kernel<DT, false, 256>;
}

int launch_kq(const w4a16_gemm_args* a, const Plan& pl, hipStream_t stream) {
  const bool zp = a->b_zeros != nullptr, channel = pl.gm == GM_CHANNEL, priv = pl.tn == 128;
  const int parts = priv ? 8 : pl.mb == 4 ? 4 : 2, wn = pl.tn / 128;
  const int period = priv ? 4 : 4 * parts;  // splits are whole multiples of so many k-steps
  const bool f16 = a->dtype == DT_F16;
  const bool short_groups = !channel && pl.group_ksteps < 4;
  const kq_fn fn = f16 ? pick_kq<DT_F16>(pl.mb, pl.tn, zp, channel, short_groups) : pick_kq<DT_BF16>(pl.mb, pl.tn, zp, channel, short_groups);
  if ((a->wtype != W4A16_WTYPE_U4B8 && a->wtype != W4A16_WTYPE_U4) || (a->flags & (W4A16_F_ZP_FLOAT | W4A16_F_MOE)) ||
      pl.gm == GM_GIDX || pl.use_perm || pl.splits < 1 || (int64_t)pl.kps * pl.splits < pl.total_ksteps ||
      pl.kps * (pl.splits - 1) >= pl.total_ksteps || pl.kps % period != 0 || pl.total_ksteps % period != 0 ||
      (pl.tn != 256 && !priv) || !fn || (priv && (a->lda < 0 || a->lda * 2 * pl.bm >= (1LL << 31))))
    return fail(W4A16_EINVAL, "unsupported kernel variant");
  const int smem = kq_smem(pl.mb, parts, wn);
  KParams p = make_kparams(a, pl);
  if (pl.tiles <= 0) return 0;
  W4A16_HIP(allow_dynamic_lds((const void*)fn, smem));
  hipLaunchKernelGGL(fn, dim3((unsigned)((int64_t)pl.tiles * pl.splits)), dim3(64 * wn * parts), smem, stream, p);
  W4A16_HIP(hipGetLastError());
  if (pl.splits > 1) {
    const kq_reduce_fn red = f16 ? pick_kq_reduce<DT_F16>(pl.tn, pl.mb, channel) : pick_kq_reduce<DT_BF16>(pl.tn, pl.mb, channel);
    hipLaunchKernelGGL(red, dim3((unsigned)pl.tiles * pl.mb), dim3(256), 0, stream, p, pl.mb);
    W4A16_HIP(hipGetLastError());
  }
  return 0;
}

}  // namespace w4a16
