// Launch plan shared between the host entry point and the kernel launchers.
#pragma once
#include "gemm_common.h"

namespace w4a16 {

struct Plan {
  int gm;            // GM_*: how scale rows are found
  int group_ksteps;  // GM_GROUPED: group_size / 32
  bool use_perm;     // gather A columns through perm (act-order)
  bool a_by_slot = false;  // MoE: A already holds one row per sorted slot (act-order gather done in front of the GEMM)
  int mb, bm;        // m-blocks of 16 rows per tile, rows per tile
  int mtiles, ncp, tiles;
  int total_ksteps, splits, kps;  // k-steps of 32 rows; K splits; k-steps per split
  int xcd_map;
  int kind;  // 0: skinny kernel, 1: decode kernel, 2: prefill ("fat") kernel, 3: 64-row ("mid") kernel,
             // 5: in-workgroup K split (gemm_kq.hip): 64 x 256 tiles in K quarters (mb = 4), 80 .. 128 x 256 in halves (mb = 5 .. 8), 32 .. 64 x 128
             // in eighths (mb = 2 .. 4, tn = 128), 6: 8-bit matrix unit, 7: the same on prepared weights,
             // 8: MoE blocks of 64 slots, integer 4-bit weights (gemm_slots.hip, tn = 256 or 512), 9: the 8-bit unit on MoE blocks of 128 slots,
             // 10: tiles of 32 or 48 rows x 64 columns, unscaled weights (gemm_rows.hip)
  int tn;    // tile width in columns (128; the decode kernel also has 64)
  int nw = 8;  // 16-row tiles (decode kernel, general kernel with one m-block): wavefronts per workgroup (8 or 4)
  int strip0 = 0;      // 64-row kernel / K-split kernel: first 512- / 256-column strip handled by the launch
  int resident = 0;    // MoE blocks of 64 slots: workgroups that run at a time
  int dyn_slots = 0;   // 64-row kernel, MoE: resident workgroups that the device-side K split of the tail tiles fills
  int tail_strips = 0; // prefill plan: trailing 512-column strips handed to another kernel (0 = none)
  int tail_kind = 3;   // ... which one: 3 = 64-row kernel, 5 = tall tiles with the K halves inside the workgroup
  int tail_mb = 8;     // ... of so many m-blocks
  int ks = 1;          // 8-bit-unit kernels: K parts inside a workgroup
  int64_t x8_bytes = 0;  // 8-bit-unit kernels: the activations split in two 8-bit terms (and the prepared weights), behind the other scratch
  int64_t ctmp_bytes;  // fp32 split-K partials
  int64_t atmp_bytes;  // column-permuted copy of A (act-order), after the partials; MoE: one row per sorted slot
};

// MoE act-order: out[slot, :] = a[sorted_ids[slot] / top_k, perm[expert of the slot's block][:]] for the valid slots
// (gemm.hip runs it in front of the GEMM kernels, which then read row `slot`).
int moe_gather_rows(const w4a16_gemm_args* a, void* out, hipStream_t stream);

// 64-row kernel, MoE: upper bound of the tail pieces (tail_split) for a launch of `tiles` tiles at most
inline int64_t mid_tail_pieces(int64_t tiles, int slots) { return tiles * 8 < slots ? tiles * 8 : slots; }

int launch_skinny(const w4a16_gemm_args* a, const Plan& pl, hipStream_t stream);
int launch_rows(const w4a16_gemm_args* a, const Plan& pl, hipStream_t stream);
int launch_decode(const w4a16_gemm_args* a, const Plan& pl, hipStream_t stream);
int launch_fat(const w4a16_gemm_args* a, const Plan& pl, hipStream_t stream);
int launch_mid(const w4a16_gemm_args* a, const Plan& pl, hipStream_t stream);
// What a plan may ask for beyond partial tiles and copies of A that other plans need too: prepared weights, and the terms of MoE rows (two bytes for
// each slot and element, where the 16-bit kernels read A in place).  8 experts of 4096 x 14336, top-2, 4096 tokens: 251 MiB; 8192 x 57344: 448.
constexpr int64_t X8_EXTRA_MAX = 512LL << 20;
int64_t x8_scratch_bytes(int64_t rows, int64_t k);
int64_t x8_weight_bytes(int64_t k, int64_t n);
int64_t x8_moe_scratch_bytes(int64_t n_sorted, int64_t k);
int launch_x8_moe(const w4a16_gemm_args* a, const Plan& pl, void* scratch, hipStream_t stream);
int launch_x8(const w4a16_gemm_args* a, const Plan& pl, void* scratch, hipStream_t stream);
int launch_slots(const w4a16_gemm_args* a, const Plan& pl, hipStream_t stream);
int launch_kq(const w4a16_gemm_args* a, const Plan& pl, hipStream_t stream);

}  // namespace w4a16
