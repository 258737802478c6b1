// W4A16 GEMM for gfx950, MoE blocks of 64 sorted token slots, integer 4-bit weights: tiles of 64 rows x 256 or 512 columns
// (the counterpart of the reference's thread_m_blocks = 4 configurations, csrc/moe/marlin_moe_wna16/ops.cu:451-512).
//
//   4 wavefronts, each owning 64 rows x 64 (W = 2) or 128 (W = 4) columns, operands in registers: A from LDS, double buffered, weights streamed
//   global -> registers four k-steps ahead and dequantised between the MFMAs, as in the 64-row kernel (gemm_mid.hip).  What differs, and why:
//   narrow tiles   the 512-column tiles of that kernel are few where experts are small or hold few rows (16 experts of 1024 x 2048: 64 and 32
//                  tiles on 512 workgroups), and two of them fill the registers of a compute unit.  Half the columns need fewer than 170 registers
//                  (accumulators among them, and no accumulation registers: their split would halve the rest), so three workgroups share a unit.
//                  The price is that A is read twice as often; it pays until the 512-column tiles alone fill their workgroups (see the planner).
//   live m-blocks  a block's rows stand in front: with r of them only ceil(r / 16) m-blocks are multiplied and stored.  The loop exists once per
//                  number of m-blocks; the weights it streams are the same, so this saves up to 3/4 of the matrix and LDS work, not of the loads.
//   buffer loads   uniform base and row in scalar registers, one 32-bit offset per lane: no address arithmetic on the VALU, which bounds the loop,
//                  and the registers of the addresses.  So both operands stay under 2 GiB (the planner checks; gemm_mid.hip takes the others).
// Measured, whole layers in a graph (7 expert shapes of 1024 x 2048 to 4096 x 14336, 12 to 192 slots per expert, even and skewed routing, fp16 and
// bf16, groups of 32 to channel-wise; 945 layers): 0.87 of the time on 512-column tiles of the 64-row kernel in the mean, 0.70 - 0.85 with small
// experts or few rows, 0.95 - 1.02 with full blocks and many tiles.  128 experts of 2048 x 768, top-8, 601 tokens, bf16 AWQ: layer 124.3 -> 118.8 us (112 with what came
// later: scalar loads in front of the loop, rows read together behind it, priorities, and the launches around the GEMMs).
// Requirements (host-checked): MoE blocks of 64 slots, K % 128 == 0, power-of-two groups or one scale per column, A's columns in weight order.
#include <type_traits>

#include "gemm_kernels.h"

namespace w4a16 {

constexpr int SL_BM = 64;
constexpr int SL_D = 4;  // weight k-steps in flight per wavefront
// dwords of one k-step of an A buffer: four m-blocks x 64 lanes x 16 B, and half a row of the LDS banks (staging stores, see kq_kstep)
constexpr int SL_KSTEP = 4 * 256 + 32;
constexpr int SL_ABUF = 2 * SL_KSTEP * 4;    // one A buffer: 2 k-steps
// Cutting a tail in two (see tail_split) costs its partial tiles and the second pass: it gains where the halves are long.  Two pieces over none, tails
// of 0.4 to 0.5 of the workgroups: W = 2 K = 3072 0.95 - 1.02, 4096 0.91 - 0.98, 7168 0.95 - 0.98, 14336 0.79; W = 4 K = 3072 1.02 - 1.06,
// 4096 1.00 - 1.08, 6144 0.98, 7168 0.86 - 0.99, 14336 0.91.
constexpr int sl_min_split(int w, int total_ksteps) { return total_ksteps >= (w == 2 ? 128 : 192) ? 2 : 3; }
constexpr int sl_rs(int w) { return w == 4 ? RED_RS : 76; }  // floats per row of an epilogue slab: two halves of 16 w columns and 8 between them
constexpr int sl_smem(int w) {
  const int slabs = 4 * 16 * sl_rs(w) * 4;
  return (2 * SL_ABUF > slabs ? 2 * SL_ABUF : slabs) + SL_BM * 8;  // + C row and routing weight of each tile row
}
// Tile j of the launch's first `tiles` ones: workgroup b runs on XCD b mod 8, which gets a contiguous run of them
__device__ __forceinline__ int xcd_run(int j, int tiles) {
  const int xcd = j & 7, rem = tiles & 7;
  return xcd * (tiles >> 3) + min(xcd, rem) + (j >> 3);
}
template <int W>
using uvec = uint32_t __attribute__((ext_vector_type(W)));
template <int W>
__device__ __forceinline__ uvec<W> load_words(__amdgpu_buffer_rsrc_t res, uint32_t off, uint32_t soff) {
  if constexpr (W == 4)
    return __builtin_bit_cast(uvec<W>, __builtin_amdgcn_raw_buffer_load_b128(res, off, soff, 0));
  else
    return __builtin_bit_cast(uvec<W>, __builtin_amdgcn_raw_buffer_load_b64(res, off, soff, 0));
}

// ONCE: scale groups of 128 rows at least, or one scale per column: constants made once per loop iteration
// W: Marlin words of a lane; a wavefront owns 32 W columns, a tile 128 W
template <int DT, bool ZP, bool CHANNEL, bool ONCE, int W>
__global__ __launch_bounds__(256, W == 2 ? 3 : 2) void slots_kernel(const KParams p) {
  static_assert(W == 2 || W == 4, "256 or 512 columns");
  constexpr int TN = 128 * W, RS = sl_rs(W), SMEM = sl_smem(W), HALF = 16 * W, AD = 2;  // HALF: columns of either n-tile (or half of one)
  constexpr bool UNIT = CHANNEL;
  extern __shared__ __align__(16) unsigned char smem[];
  int* s_crow = (int*)(smem + SMEM - SL_BM * 8);
  float* s_tw = (float*)(smem + SMEM - SL_BM * 4);
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int c = lane & 7, h = (lane >> 3) & 1, g = lane >> 4;

  // The chain in front of the first weights: arguments, number of live slots, the tile's expert and slot ids, its rows and weights.  So the arguments are
  // asked for together, and the number and the expert are scalar loads (the compiler makes one of the first as long as nothing has been stored: the side
  // job stands behind it, in front of every exit).  (Asked for one by one as they are used: 4.2 us to the first products, of 60; 128
  // experts of 2048 x 768, top-8, 601 and 1300 tokens 119.7 -> 117.6 and 199.5 -> 189.9 us, five other layers 1.00.)
  const int moe_ntp = *p.ntpp;
  asm volatile("" ::"s"(p.A), "s"(p.B), "s"(p.S), "s"(p.sorted_ids), "s"(p.expert_ids), "s"(p.b_estride), "s"(p.s_estride), "s"(p.N), "s"(p.K), "s"(p.ncp),
               "s"(p.top_k), "s"(p.c_rows), "s"(p.total_ksteps), "s"(p.dyn_slots), "s"(p.group_shift));
  const int mtiles = (p.n_sorted + SL_BM - 1) / SL_BM;
  const int live = min((moe_ntp + SL_BM - 1) / SL_BM, mtiles);
  if (live == 0) {
    zero_fill_side_job(p);
    return;
  }
  int j = blockIdx.x, split = 0, nsplit = 1, kps = p.total_ksteps, tile = 0, mt, strip;
  // live tiles: whole ones in runs for every XCD, then the pieces along K of those of the last, partly filled round (see tail_split), which walk
  // the tiles first, then K; a short K is never cut
  const TailSplit d = p.dyn_slots > 0 ? tail_split(live * p.ncp, p.dyn_slots, p.total_ksteps, sl_min_split(W, p.total_ksteps)) : TailSplit{live * p.ncp, 0, 1, p.total_ksteps};
  if (j < d.F) {
    j = xcd_run(j, d.F);
  } else {
    const int u = j - d.F;
    if (u >= d.R * d.S) {
      zero_fill_side_job(p);
      return;
    }
    tile = u % d.R, split = u / d.R, nsplit = d.S, kps = d.kps;
    j = d.F + tile;
  }
  chunked_tile(j, live, p.ncp, mt, strip);
  const int row0 = mt * SL_BM;
  const bool act = p.act;
  // W = 4: a column pair u, two n-tiles (lanes h = 0 / 1), all their words; with the fused SiLU-and-mul gate n-tile u and its up n-tile.
  // W = 2: an n-tile u (lanes h = 0 / 1: its first / last 32 columns, words 2h and 2h + 1), or 32 columns of gate n-tile u / 2 and the same of
  // its up n-tile (words 2 (u & 1) and the next of either).
  const int u = strip * 4 + wv;
  const bool wave_on = u * (2 * HALF) < p.N;  // trailing wavefronts only help staging

  const uint32_t* Bq = p.B;
  const uint16_t* Sc = (const uint16_t*)p.S;
  const uint32_t* Zp = p.Z;
  const uint16_t* bias = (const uint16_t*)p.bias;
  {
    int e;
    asm volatile("s_load_dword %0, %1, %2\n\ts_waitcnt lgkmcnt(0)" : "=&s"(e) : "s"(p.expert_ids), "s"(mt * 4));
    zero_fill_side_job(p);
    if (e < 0) return;  // expert of another rank
    Bq += e * p.b_estride;
    Sc += e * p.s_estride;
    if (ZP) Zp += e * p.z_estride;
    if (bias) bias += e * p.n_estride;
  }
  // which A row feeds tile row r and which C row receives it (-1: none)
  auto tile_row_ids = [&](int r, int& src, int& dst) {
    src = dst = -1;
    const int id = row0 + r < p.n_sorted ? p.sorted_ids[row0 + r] : -1;
    if ((unsigned)id < (unsigned)p.c_rows) {
      src = p.a_by_slot ? row0 + r : id / p.top_k;
      dst = id;
    }
  };
  // m-blocks that hold a row (rows without one stand behind them: their products are left out)
  int live_mb;
  {
    int src, dst;
    tile_row_ids(lane, src, dst);
    const uint64_t rows = __ballot(dst >= 0);
    if (rows == 0) return;
    live_mb = (79 - __builtin_clzll(rows)) >> 4;
    if (wv == 0) {
      s_crow[lane] = dst;
      // (read here once: in the epilogue a load per row would wait behind every store in front of it)
      if (p.mul_topk) s_tw[lane] = dst >= 0 ? p.topk_w[dst] : 0.f;
    }
  }

  // ---- weights of this wavefront
  const int nt = !wave_on ? 0
                 : W == 4 ? (act ? (h ? p.N >> 7 : 0) + u : (2 * u + h) * 64 < p.N ? 2 * u + h : 2 * u)
                          : act ? (h ? p.N >> 7 : 0) + (u >> 1) : u;
  const int word0 = W == 4 ? 0 : act ? 2 * (u & 1) : 2 * h;
  // buffer resources: uniform bases and 32-bit offsets, nothing per lane but the lane's own (the host checks the sizes)
  const uint32_t b_row = (uint32_t)p.N * 8;  // bytes of one k-tile
  const int sg = CHANNEL ? 1 : p.total_ksteps >> p.group_shift;
  const auto a_res = __builtin_amdgcn_make_buffer_rsrc((void*)p.A, 0, 0x7fffffff, 0x00020000);
  const auto b_res = __builtin_amdgcn_make_buffer_rsrc((void*)Bq, 0, (int)((uint32_t)(p.K / 16) * b_row), 0x00020000);
  const auto s_res = __builtin_amdgcn_make_buffer_rsrc((void*)Sc, 0, sg * p.N * 2, 0x00020000);
  const auto z_res = __builtin_amdgcn_make_buffer_rsrc((void*)Zp, 0, sg * (p.N / 2), 0x00020000);
  const uint32_t b_off = (uint32_t)(nt * 128 + (4 * c + g) * 4 + word0) * 4;
  // (nt * 64 + 8 c + 2 word0) * 2 of the scales, (nt * 8 + c) * 4 of the zero points and the shift to word0's: made from b_off when they are
  // wanted, two instructions per use for three of the loop's registers
  auto from_b = [&](auto shift_tag) {
    uint32_t v;
    asm volatile("v_lshrrev_b32 %0, %2, %1" : "=v"(v) : "v"(b_off), "n"(decltype(shift_tag)::value));
    return v;
  };
  auto s_off = [&]() { return (from_b(std::integral_constant<int, 2>{}) & ~15u) + (b_off & 8u); };
  auto z_off = [&]() { return from_b(std::integral_constant<int, 4>{}) & ~3u; };

  // ---- activation staging: thread t loads piece (t & 7) of tile rows (t >> 3) + 32 i, i = 0..1
  // (rows without a source read row 0 of A; their results are never stored)
  const int piece = t & 7;
  uint32_t a_off[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    int src, dst;
    tile_row_ids((t >> 3) + 32 * i, src, dst);
    a_off[i] = (uint32_t)(src < 0 ? 0 : src) * ((uint32_t)p.lda * 2) + piece * 16;
  }
  // LDS A layout: [buffer][k-step 2][m-block 4][lane 64][4 dwords]; the 16 bytes of (row, piece) are the K
  // pairs 8*pp + 2q (pp = piece & 3), which belong to lane (q*16 + row%16), dword pp, of k-step piece >> 2.
  uint32_t* lds = (uint32_t*)smem;
  const int a_wr = (piece >> 2) * SL_KSTEP + ((t >> 7) * 64 + ((t >> 3) & 15)) * 4 + (piece & 3);
  // AD half chunks in flight, each stored AD k-steps after its load.  (Loads return in order: waiting for one waits for the weights asked for in front
  // of it, so this is also how many k-steps those have.  One: 1.03 of the time at W = 2, 1.01 at W = 4; four, which spills: 0.995.)
  u32x4 areg[AD];
  // this workgroup's k-steps: [ks_b, ks_e), a multiple of 4 long (the host splits K in multiples of 4 k-steps)
  const int ks_b = split * kps;
  const int ks_e = min(ks_b + kps, p.total_ksteps);
  auto load_a = [&](int c0, auto half_tag) {  // half chunk: half & 1 of chunk c0 + half / 2, relative to ks_b
    constexpr int H = decltype(half_tag)::value;
    const int chunk = ks_b / 2 + c0 + H / 2;
    areg[H % AD] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(a_res, a_off[H & 1], (uint32_t)chunk * 128, 0));
  };
  auto store_a = [&](auto half_tag) {
    constexpr int H = decltype(half_tag)::value;
    uint32_t* dst = lds + (H / 2 & 1) * (SL_ABUF / 4) + a_wr + (H & 1) * 512;
#pragma unroll
    for (int q = 0; q < 4; ++q) dst[q * 64] = areg[H % AD][q];
  };
#define HALF_CHUNK(h) std::integral_constant<int, (h)>{}

  struct Stage {
    uvec<W> b0, b1, sc;
    uint32_t zq;
  };
  Stage st[SL_D];
  uvec<W> sc128 = {};
  uint32_t zq128 = 0;
  auto issue_scales = [&](int ks) {
    const uint32_t gi = CHANNEL ? 0 : (ks_b + ks) >> p.group_shift;
    if (!CHANNEL) sc128 = load_words<W>(s_res, s_off(), gi * p.N * 2);
    if (ZP) zq128 = __builtin_amdgcn_raw_buffer_load_b32(z_res, z_off(), gi * (p.N / 2), 0);
  };
  auto issue = [&](Stage& s, int ks) {  // ks: relative to ks_b
    ks += ks_b;
    if constexpr (!ONCE) {
      const uint32_t gi = ks >> p.group_shift;  // (power-of-two groups: host)
      s.sc = load_words<W>(s_res, s_off(), gi * p.N * 2);
      if (ZP) s.zq = __builtin_amdgcn_raw_buffer_load_b32(z_res, z_off(), gi * (p.N / 2), 0);
    }
    s.b0 = load_words<W>(b_res, b_off, (uint32_t)(2 * ks) * b_row);
    s.b1 = load_words<W>(b_res, b_off, (uint32_t)(2 * ks + 1) * b_row);
  };
  auto col_const = [&](const Stage& s, int w) {
    const uint32_t zq = ONCE ? zq128 : s.zq;
    return make_col_const<DT, UNIT>(CHANNEL ? 0u : ONCE ? sc128[w] : s.sc[w], ZP ? zero_pair(W == 4 ? zq : zq >> (b_off & 8u), w) : ZERO_U4B8);
  };

  // the tile with LIVE m-blocks, to its end (so that its accumulators are not those of another loop)
  auto run = [&](auto live_tag) __attribute__((always_inline)) {
    constexpr int LIVE = decltype(live_tag)::value;
    f32x4 acc[LIVE][W][2];
#pragma unroll
    for (int mb = 0; mb < LIVE; ++mb)
#pragma unroll
      for (int w = 0; w < W; ++w) {
        acc[mb][w][0] = f32x4{0, 0, 0, 0};
        acc[mb][w][1] = f32x4{0, 0, 0, 0};
      }

    const int nchunks = (ks_e - ks_b) / 2;  // even: K % 128 == 0 and splits are multiples of 4 k-steps

    // ---- prologue
    load_a(0, HALF_CHUNK(0));
    load_a(0, HALF_CHUNK(1));
    if constexpr (ONCE) issue_scales(0);
#pragma unroll
    for (int j = 0; j < SL_D; ++j) issue(st[j], j);
    store_a(HALF_CHUNK(0));
    store_a(HALF_CHUNK(1));
    load_a(0, HALF_CHUNK(2));
    // B operands of two Marlin words: the one whose MFMAs are being issued and the one being dequantised
    u32x4 ob[2][2];
    ColConst<DT> ccs[W];
#pragma unroll
    for (int w = 0; w < W; ++w)
      if (ONCE || w == 0) ccs[w] = col_const(st[0], w);
    dequant_pair<DT, UNIT>(st[0].b0[0], st[0].b1[0], ccs[0], ob[0][0], ob[0][1]);
    __syncthreads();

    // One k-step: per word, 2 LIVE MFMAs on ob[w & 1], column half 0 first (its registers are free for the next word's half 1); between them the
    // eight registers of the following word's operands (word w + 1 of this k-step, or word 0 of the next k-step `nxt`) are made into
    // ob[(w + 1) & 1], in three dependent steps each, of which three consecutive registers are at one step each (see gemm_kq.hip).
    auto a_frags = [&](int buf, int kk) { return (const u32x4*)(lds + buf * (SL_ABUF / 4) + kk * SL_KSTEP) + lane; };
    // EARLY: the A operands of the next k-step are read during this one's last word, each behind the last MFMA that uses its registers, and the next
    // chunk is stored and the barrier passed before that.  Layers of 64 to 192 slots per expert 0.97 of the time; with one or two m-blocks a
    // word is over before the reads are (1.00).
    constexpr bool EARLY = LIVE > 2;
    u32x4 af[LIVE];
    if constexpr (EARLY) {
#pragma unroll
      for (int mb = 0; mb < LIVE; ++mb) af[mb] = a_frags(0, 0)[mb * 64];
    }
    // store_tag: the half chunk that the chunk's second k-step stores, 0 in its first
    auto kstep = [&](int buf, auto store_tag, const Stage& cur, const Stage& nxt, auto refresh_tag, auto end_tag) __attribute__((always_inline)) {
      constexpr bool REFRESH = decltype(refresh_tag)::value, KK = decltype(store_tag)::value > 0;
      const u32x4* anext = KK ? a_frags(buf ^ 1, 0) : a_frags(buf, 1);
      if constexpr (!EARLY) {
#pragma unroll
        for (int mb = 0; mb < LIVE; ++mb) af[mb] = a_frags(buf, KK)[mb * 64];
      }
      if constexpr (!ONCE) ccs[1] = col_const(cur, 1);
      uint32_t halves = 0;
      PieceValue<DT> value;
      auto make_halves = [&](auto p_tag) {  // register P of the k-step: J = P & 7 of the word behind word P >> 3
        constexpr int P = decltype(p_tag)::value, G = P >> 3, J = P & 7, NW = (G + 1) % W;
        const Stage& src = G == W - 1 ? nxt : cur;
        halves = piece_halves<J>((J & 3) < 2 ? src.b0[NW] : src.b1[NW]);
      };
      make_halves(std::integral_constant<int, 0>{});
      value = piece_value<DT, 0>(halves, ccs[1]);
      make_halves(std::integral_constant<int, 1>{});
      for_each_piece<8 * W>([&](auto p_tag) __attribute__((always_inline)) {
        constexpr int P = decltype(p_tag)::value, w = P >> 3, J = P & 7, NW = (w + 1) % W;
        if constexpr (EARLY && KK && P == 8 * W - 12 && !decltype(end_tag)::value) store_a(store_tag);
        if constexpr (EARLY && KK && P == 8 * W - 4) __syncthreads();
        if constexpr (decltype(end_tag)::value && P == 8 * W - 8) {  // (nothing is made behind the last operands: see apart below)
          asm volatile("s_nop 1");
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int i = J * LIVE / 4; i < (J + 1) * LIVE / 4; ++i) {
          mfma_inplace_v<DT>(acc[i % LIVE][w][i / LIVE], af[i % LIVE], ob[w & 1][i / LIVE]);
          if (EARLY && w == W - 1 && i >= LIVE) af[i % LIVE] = anext[(i % LIVE) * 64];
        }
        ob[NW & 1][J >> 2][J & 3] = piece_finish<DT, UNIT, J>(value, ccs[NW]);
        // the constants the next registers want, each as soon as the old ones have been used
        if constexpr (ONCE) {
          if constexpr (REFRESH && w == W - 2 && J == 4) ccs[0] = col_const(nxt, 0);
          if constexpr (REFRESH && w == W - 1 && J == 1) ccs[1] = col_const(nxt, 1);
          if constexpr (REFRESH && W == 4 && w == W - 1 && J == 3) ccs[W - 2] = col_const(nxt, W - 2);
          if constexpr (REFRESH && W == 4 && w == W - 1 && J == 5) ccs[W - 1] = col_const(nxt, W - 1);
        } else if constexpr (w < W - 1 && J == 4) {
          ccs[(w + 2) % W] = col_const(w == W - 2 ? nxt : cur, (w + 2) % W);
        }
        if constexpr (P + 1 < 8 * W) value = piece_value<DT, (P + 1) & 7>(halves, ccs[(((P + 1) >> 3) + 1) % W]);
        if constexpr (P + 2 < 8 * W) make_halves(std::integral_constant<int, P + 2>{});
        __builtin_amdgcn_sched_barrier(0);
      });
    };

    auto end_chunk = [&](auto store_tag, auto end_tag) {
      if constexpr (!EARLY) {
        if constexpr (!decltype(end_tag)::value) store_a(store_tag);
        __syncthreads();
      }
    };

    Pace pace;
    pace.start(nchunks, (int)blockIdx.x + p.resident >= d.F + d.R * d.S);
    // ---- main loop: two chunks (four k-steps = the weight ring) per iteration.  The last iteration stands behind it and asks for nothing: as part of the
    // loop it read its own data again, and the epilogue's registers waited for that: 1.011 of the time in the mean of 45 layers of 8 to 128 experts, 0.972 to
    // 1.039 (both GEMMs, weights not cached; 128 experts of 2048 x 768, 601 tokens level, 1300 tokens 177.5 -> 173.5 us, 32 of 3072 x 1024, 600 tokens
    // 93.1 -> 91.0).
    auto round = [&](int c0, auto end_tag) __attribute__((always_inline)) {
      constexpr bool END = decltype(end_tag)::value;
      const int ks0 = 2 * c0;
      // (two wait states between the operands' last register and their first MFMA, where the loads' issue stands otherwise: the compiler does not see
      //  the MFMAs)
      auto apart = [] {
        if constexpr (END) {
          asm volatile("s_nop 1");
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      pace.round(c0);
      load_a(c0, HALF_CHUNK(AD + 1));
      apart();
      kstep(0, HALF_CHUNK(0), st[0], st[1], std::false_type{}, std::false_type{});
      if constexpr (ONCE && !END) issue_scales(ks0 + 4);
      if (!END) issue(st[0], ks0 + 4);
      store_a(HALF_CHUNK(2));
      if (!END) load_a(c0, HALF_CHUNK(AD + 2));
      apart();
      kstep(0, HALF_CHUNK(3), st[1], st[2], std::false_type{}, std::false_type{});
      if (!END) issue(st[1], ks0 + 5);
      end_chunk(HALF_CHUNK(3), std::false_type{});
      if (!END) load_a(c0, HALF_CHUNK(AD + 3));
      apart();
      kstep(1, HALF_CHUNK(0), st[2], st[3], std::false_type{}, std::false_type{});
      if (!END) issue(st[2], ks0 + 6);
      if (!END) store_a(HALF_CHUNK(4));
      if (!END) load_a(c0, HALF_CHUNK(AD + 4));
      apart();
      kstep(1, HALF_CHUNK(5), st[3], st[0], std::true_type{}, end_tag);
      if (!END) issue(st[3], ks0 + 7);
      end_chunk(HALF_CHUNK(5), end_tag);
    };
#pragma unroll 1
    for (int c0 = 0; c0 < nchunks - 2; c0 += 2) round(c0, std::false_type{});
    round(nchunks - 2, std::true_type{});
#undef HALF_CHUNK

    // ------------------------------------------------------------------------------ epilogue
    // (the inline-asm MFMAs are opaque to the compiler's hazard logic: let the matrix pipe drain before the
    //  accumulators are read)
    asm volatile("s_nop 15\n\ts_nop 15\n\ts_nop 15" ::: "memory");
    // per wavefront and m-block: accumulators -> private LDS slab [16 rows][RS] -> 8-byte row stores.  All rows of an m-block are read before one is
    // stored: read and stored one by one, each read was waited for by itself (GEMM2 of 128 experts: 6 us of 40 behind the loop).
    // (the last barrier of the loop separates the slabs from the A buffers they overlay)
    if (!wave_on) return;
    int el = lane;  // (a lane's places are worked out again here: kept through the loop they would spill)
    asm volatile("" : "+v"(el));
    float* slab = (float*)smem + wv * (16 * RS);
    const int slab_at = 4 * (el >> 4) * RS + (HALF + 8) * (el >> 3 & 1) + (el & 7);
    // 8 W lanes to a row: columns lc .. + 3 of the wavefront's 32 W; fused SiLU-and-mul, unsplit, 4 W lanes: gate columns ac .. + 3 of the first
    // HALF and the up columns of the same outputs
    constexpr int LR = 8 * W, LA = 4 * W;
    const int lc = (el % LR) * 4, lpos = lc / HALF * (HALF + 8) + lc % HALF, ac = (el % LA) * 4;
    const int ncol = 2 * HALF * u + lc, ocol = HALF * u + ac;
    const int er = el / LR;  // first row of the lane
    if (!act && ncol >= p.N) el = -1;  // (the second n-tile of the last pair may be missing)
    float cs[4] = {1.f, 1.f, 1.f, 1.f}, bs[4] = {0.f, 0.f, 0.f, 0.f}, cu[4] = {1.f, 1.f, 1.f, 1.f}, bu[4] = {0.f, 0.f, 0.f, 0.f};
    auto col_consts = [&](int col, float* sc_out, float* b_out) {
      const int base = col & ~31, cl = col & 31;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (CHANNEL) sc_out[j] = lo_f32<DT>(Sc[base + single_perm_pos(cl + j)]);
        if (bias) b_out[j] = lo_f32<DT>(bias[base + single_perm_pos(cl + j)]);
      }
    };
    if (act) {
      col_consts(ocol, cs, bs);
      col_consts((p.N >> 1) + ocol, cu, bu);
    } else if (el >= 0) {
      col_consts(ncol, cs, bs);
    }
#pragma unroll
    for (int mb = 0; mb < LIVE; ++mb) {
#pragma unroll
      for (int w = 0; w < W; ++w)
#pragma unroll
        for (int hf = 0; hf < 2; ++hf)
#pragma unroll
          for (int r = 0; r < 4; ++r) slab[slab_at + r * RS + 16 * w + 8 * hf] = acc[mb][w][hf][r];
      __builtin_amdgcn_wave_barrier();
      if (act && nsplit == 1) {
        constexpr int NI = 16 * LA / 64;
        f32x4 v[NI], up[NI];
        int crow[NI];
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          const int r16 = el / LA + 64 / LA * i;
          crow[i] = s_crow[mb * 16 + r16];
          v[i] = *(const f32x4*)(slab + r16 * RS + ac);
          up[i] = *(const f32x4*)(slab + r16 * RS + ac + HALF + 8);
        }
#pragma unroll
        for (int i = 0; i < NI; ++i) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            v[i][j] = v[i][j] * cs[j] + bs[j];
            up[i][j] = up[i][j] * cu[j] + bu[j];
          }
          if (p.mul_topk) {
            const float tw = s_tw[mb * 16 + el / LA + 64 / LA * i];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              v[i][j] *= tw;
              up[i][j] *= tw;
            }
          }
          if (crow[i] >= 0) store_row4_silu_mul<DT>(p, crow[i], ocol, v[i], up[i]);
        }
        __builtin_amdgcn_wave_barrier();
        continue;
      }
      constexpr int NI = 16 * LR / 64;
      f32x4 rows[NI];
      int crows[NI];
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int r16 = er + 64 / LR * i;
        crows[i] = s_crow[mb * 16 + r16];
        rows[i] = *(const f32x4*)(slab + r16 * RS + lpos);
      }
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int r16 = er + 64 / LR * i, crow = crows[i];
        f32x4 v = rows[i];
        if (el < 0 || crow < 0) continue;
        if (nsplit > 1) {
          // K is split: the fp32 partial tile [row 64][column TN] goes to scratch; the kernel launched behind this one adds the
          // splits and finishes the rows
          *(f32x4*)(p.ctmp + (((int64_t)tile * nsplit + split) * SL_BM + mb * 16 + r16) * TN + wv * (2 * HALF) + lc) = v;
          continue;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = v[j] * cs[j] + bs[j];
        if (p.mul_topk) {
          const float tw = s_tw[mb * 16 + r16];
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] *= tw;
        }
        store_row4<DT>(p, crow, ncol, v);
      }
      __builtin_amdgcn_wave_barrier();
    }
  };
  if (live_mb == 4)
    run(std::integral_constant<int, 4>{});
  else if (live_mb == 3)
    run(std::integral_constant<int, 3>{});
  else if (live_mb == 2)
    run(std::integral_constant<int, 2>{});
  else
    run(std::integral_constant<int, 1>{});
}

// Second pass: adds the pieces of the tail tiles in K order and finishes the rows as the kernel itself does.  One workgroup per (tile, 16-row
// block); thread -> 4 columns of every (8 / W)-th row.
template <int DT, bool CHANNEL, int W>
__global__ __launch_bounds__(256) void slots_reduce_kernel(const KParams p) {
  constexpr int TN = 128 * W, HALF = 16 * W, TR = TN / 4;  // TR: threads to a row
  const int t = threadIdx.x;
  const int mtiles = (p.n_sorted + SL_BM - 1) / SL_BM;
  const int tile = blockIdx.x / 4, rb = blockIdx.x % 4;  // tile: index among the tail tiles (see tail_split)
  const int live = min((*p.ntpp + SL_BM - 1) / SL_BM, mtiles);
  if (live == 0) return;
  const TailSplit d = tail_split(live * p.ncp, p.dyn_slots, p.total_ksteps, sl_min_split(W, p.total_ksteps));
  if (d.S == 1 || tile >= d.R) return;
  const int nsplit = d.S;
  int mt, strip;
  chunked_tile(d.F + tile, live, p.ncp, mt, strip);
  const int row0 = mt * SL_BM;
  const uint16_t* Sc = (const uint16_t*)p.S;
  const uint16_t* bias = (const uint16_t*)p.bias;
  const int e = p.expert_ids[mt];
  if (e < 0) return;
  Sc += e * p.s_estride;
  if (bias) bias += e * p.n_estride;
  const bool act = p.act;
  const int fc4 = (t % TR) * 4, u = strip * 4 + fc4 / (2 * HALF), cl = fc4 % (2 * HALF);
  // fused SiLU-and-mul: a wavefront's 32 W columns are HALF gate columns and the up columns of the same outputs
  const int ncol = act ? HALF * u + cl : 2 * HALF * u + cl;
  if (act ? u * 2 * HALF >= p.N || cl >= HALF : ncol >= p.N) return;
  float cs[4] = {1.f, 1.f, 1.f, 1.f}, bs[4] = {0.f, 0.f, 0.f, 0.f}, cu[4] = {1.f, 1.f, 1.f, 1.f}, bu[4] = {0.f, 0.f, 0.f, 0.f};
  auto col_consts = [&](int col, float* sc_out, float* b_out) {
    const int base = col & ~31, cl32 = col & 31;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (CHANNEL) sc_out[j] = lo_f32<DT>(Sc[base + single_perm_pos(cl32 + j)]);
      if (bias) b_out[j] = lo_f32<DT>(bias[base + single_perm_pos(cl32 + j)]);
    }
  };
  col_consts(ncol, cs, bs);
  if (act) col_consts((p.N >> 1) + ncol, cu, bu);
  const float* parts = p.ctmp + (int64_t)tile * nsplit * (SL_BM * TN) + fc4;
  // (the rows' slot ids, then per row the partial tiles of four splits at a time, are loaded together: the pass is bound
  //  by round trips, not by bytes)
  constexpr int NR = 16 * TR / 256;
  int crows[NR];
  float tws[NR];
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int r = rb * 16 + t / TR + 256 / TR * i;
    const int id = row0 + r < p.n_sorted ? p.sorted_ids[row0 + r] : -1;
    crows[i] = (unsigned)id < (unsigned)p.c_rows ? id : -1;
  }
#pragma unroll
  for (int i = 0; i < NR; ++i) tws[i] = (p.mul_topk && crows[i] >= 0) ? p.topk_w[crows[i]] : 1.0f;
  auto sum_splits = [&](const float* src) {  // src: the row's columns in split 0; added in split order
    f32x4 sum = {0, 0, 0, 0};
    for (int s0 = 0; s0 < nsplit; s0 += 4) {
      f32x4 a[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) a[q] = *(const f32x4*)(src + (int64_t)min(s0 + q, nsplit - 1) * (SL_BM * TN));
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (s0 + q < nsplit) sum += a[q];
    }
    return sum;
  };
#pragma unroll 2
  for (int i = 0; i < NR; ++i) {
    const int r = rb * 16 + t / TR + 256 / TR * i;
    const int crow = crows[i];
    if (crow < 0) continue;
    f32x4 v = sum_splits(parts + (int64_t)r * TN), up = {0, 0, 0, 0};
    if (act) up = sum_splits(parts + (int64_t)r * TN + HALF);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[j] = v[j] * cs[j] + bs[j];
      up[j] = up[j] * cu[j] + bu[j];
    }
    if (p.mul_topk) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[j] *= tws[i];
        up[j] *= tws[i];
      }
    }
    if (act)
      store_row4_silu_mul<DT>(p, crow, ncol, v, up);
    else
      store_row4<DT>(p, crow, ncol, v);
  }
}

typedef void (*slots_fn)(const KParams);
template <int DT, bool ZP, int W>
static slots_fn pick_slots(bool channel, bool once) {
  if (channel) return slots_kernel<DT, ZP, true, true, W>;
  return once ? slots_kernel<DT, ZP, false, true, W> : slots_kernel<DT, ZP, false, false, W>;
}
template <int DT, int W>
static slots_fn pick_slots(bool zp, bool channel, bool once) {
  return zp ? pick_slots<DT, true, W>(channel, once) : pick_slots<DT, false, W>(channel, once);
}
template <int DT, int W>
static slots_fn pick_slots_reduce(bool channel) {
  return channel ? slots_reduce_kernel<DT, true, W> : slots_reduce_kernel<DT, false, W>;
}

int launch_slots(const w4a16_gemm_args* a, const Plan& pl, hipStream_t stream) {
  const bool zp = a->b_zeros != nullptr, channel = pl.gm == GM_CHANNEL, f16 = a->dtype == DT_F16, wide = pl.tn == 512;
  const bool once = pl.group_ksteps >= 4;
  if ((a->wtype != W4A16_WTYPE_U4B8 && a->wtype != W4A16_WTYPE_U4) || (a->flags & W4A16_F_ZP_FLOAT) || !(a->flags & W4A16_F_MOE) || pl.splits != 1 ||
      pl.gm == GM_GIDX || pl.total_ksteps % 4 != 0 || (pl.tn != 256 && !wide))
    return fail(W4A16_EINVAL, "unsupported kernel variant");
  const slots_fn fn = f16 ? (wide ? pick_slots<DT_F16, 4>(zp, channel, once) : pick_slots<DT_F16, 2>(zp, channel, once))
                          : (wide ? pick_slots<DT_BF16, 4>(zp, channel, once) : pick_slots<DT_BF16, 2>(zp, channel, once));
  const KParams p = make_kparams(a, pl);
  if (pl.tiles <= 0) return 0;
  // device-side K split of the tail tiles: at most dyn_slots pieces behind the whole tiles, at most that many tail tiles
  const int64_t pieces = pl.dyn_slots > 0 ? mid_tail_pieces(pl.tiles, pl.dyn_slots) : 0;
  hipLaunchKernelGGL(fn, dim3((unsigned)(pl.tiles + pieces)), dim3(256), wide ? sl_smem(4) : sl_smem(2), stream, p);
  W4A16_HIP(hipGetLastError());
  if (pl.dyn_slots > 0) {
    const slots_fn red = f16 ? (wide ? pick_slots_reduce<DT_F16, 4>(channel) : pick_slots_reduce<DT_F16, 2>(channel))
                             : (wide ? pick_slots_reduce<DT_BF16, 4>(channel) : pick_slots_reduce<DT_BF16, 2>(channel));
    const int64_t tail = pl.tiles < pl.dyn_slots ? pl.tiles : pl.dyn_slots;
    hipLaunchKernelGGL(red, dim3((unsigned)(tail * 4)), dim3(256), 0, stream, p);
    W4A16_HIP(hipGetLastError());
  }
  return 0;
}

}  // namespace w4a16
