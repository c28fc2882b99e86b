// Tile plans of the GEMM: the tables behind tjk_gemm_plan_count / _info,
// and run_gemm, which launches one of them (gemm_kernels.h; one translation
// unit per element type).
#pragma once

#include "gemm_tiles.h"

namespace tjk {

enum { kStaged = 0, kDtl = 1, kWs = 2, kPanel = 3 };

struct GemmPlan {
  int kind, bm, bn, wm, wn, bkb, stages;
  double eff;       // prior of auto_plan's fall-back
  int ksplit = 1;   // K groups per workgroup (direct-to-LDS kernel)
  int loaders = 0;  // DMA-only waves (wave-specialized kernel)
};

// 2-byte types (bf16/fp16), BK = 64.  Which one a launch takes by default is
// gemm.hip's estimate (kAuto16); `eff` only ranks the plans where no estimated
// tile's offsets reach the rows, which leaves the staged ones (0-5).  (A 4-stage
// ring of 64-byte rows was tried and dropped: it measured 50% LDS bank-conflict
// cycles and no gain.)
static const GemmPlan kPlans16[] = {
    {kStaged, 256, 256, 2, 2, 128, 2, 0.50},  // 0
    {kStaged, 256, 128, 2, 2, 128, 2, 0.45},  // 1
    {kStaged, 128, 256, 2, 2, 128, 2, 0.45},  // 2
    {kStaged, 128, 128, 2, 2, 128, 2, 0.55},  // 3
    {kStaged, 64, 64, 2, 2, 128, 2, 0.40},    // 4
    {kStaged, 256, 256, 2, 4, 128, 2, 0.55},  // 5
    {kDtl, 256, 256, 2, 2, 128, 2, 0.85},     // 6  wave tile 128x128, 1 WG/CU
    {kDtl, 128, 128, 2, 2, 128, 2, 0.90},     // 7  wave tile 64x64, 2 WG/CU
    {kDtl, 256, 256, 2, 4, 128, 2, 1.00},     // 8  8 waves, wave tile 128x64
    {kDtl, 64, 64, 2, 2, 128, 2, 0.45},       // 9  small shapes
    {kDtl, 256, 128, 2, 2, 128, 2, 0.75},     // 10 wave tile 128x64
    {kDtl, 128, 256, 2, 2, 128, 2, 0.75},     // 11 wave tile 64x128
    {kDtl, 192, 128, 2, 2, 128, 2, 0.80},     // 12 wave tile 96x64, 1 WG/CU
    {kDtl, 192, 256, 2, 4, 128, 2, 0.90},     // 13 8 waves, wave tile 96x64
    {kDtl, 192, 384, 2, 4, 128, 2, 0.95},     // 14 8 waves, wave tile 96x96
    {kDtl, 96, 128, 1, 4, 128, 2, 0.60},      // 15 wave tile 96x32, small M
    // 16, 17: two K groups of 4 waves per workgroup (K tiles alternate between
    // the groups' LDS rings, partial sums added before the epilogue).  At the
    // packed C4 N=1024 projections they measured slower than plan 15 (FFN2
    // 60.4 vs 57.8 us): those GEMMs are partly bound by re-reading A from
    // the MALL, which splitting K does not change.
    {kDtl, 192, 128, 2, 2, 128, 2, 0.85, 2},  // 16 wave tile 96x64
    {kDtl, 128, 128, 2, 2, 128, 2, 0.85, 2},  // 17 wave tile 64x64
    // 18: a 4-slot ring (160 KB) with the spread DMA schedule, one workgroup
    // per CU.  Other deep rings measured (C4/C5 projections, residual reads
    // prefetched where registers allow) and dropped because a 2-slot plan
    // was faster on every shape: 256x256 8 waves and 4 waves with 64-byte
    // rows in 4 slots, 128x128 and 96x128 in 4 slots, 256x128 in 3 slots.
    {kDtl, 192, 128, 2, 2, 128, 4, 0.85},     // 18 wave tile 96x64, 160 KB
    // 19, 20: small tiles in deep rings (8 and 6 slots) for launches of a few
    // dozen workgroups with long K (C2's FFN2: 16 tiles, 32 K tiles each),
    // where a 2-slot ring leaves each step waiting out the DMA latency.
    {kDtl, 64, 64, 2, 2, 128, 8, 0.45},       // 19 wave tile 32x32, 128 KB
    {kDtl, 128, 64, 2, 2, 128, 6, 0.50},      // 20 wave tile 64x32, 144 KB
    // 21-23: the same small tiles with K split between 2 or 4 groups of 4
    // waves inside the workgroup (partials added through LDS), which
    // shortens the serial chain of K tiles a launch of a few dozen
    // workgroups waits out.
    {kDtl, 64, 64, 2, 2, 128, 2, 0.45, 4},    // 21 16 waves, 128 KB
    {kDtl, 64, 64, 2, 2, 128, 4, 0.45, 2},    // 22 8 waves, 128 KB
    {kDtl, 128, 64, 2, 2, 128, 3, 0.50, 2},   // 23 8 waves, 144 KB
    // 24, 25: 32-row tiles with K split between two groups of 2 / 1 waves,
    // for projections of a few hundred rows (C2: 128), whose tiles would
    // otherwise occupy a few dozen CUs each moving 128 KB of operands: at
    // 32 x 64 and 32 x 32 a launch spreads over 2x and 4x more CUs.
    {kDtl, 32, 64, 1, 2, 128, 4, 0.35, 2},    // 24 4 waves, 96 KB
    {kDtl, 32, 32, 1, 1, 128, 4, 0.30, 2},    // 25 2 waves, 64 KB
    // 26, 27: the 32-row tiles with K split between four groups, for a
    // launch of a few dozen tiles with long K (C2's FFN2, K = 2048): each
    // group streams every 4th K tile, so a workgroup has four rings' worth
    // of K tiles in flight and the serial chain is a quarter of K.
    {kDtl, 32, 32, 1, 1, 128, 4, 0.30, 4},    // 26 4 waves, 128 KB
    {kDtl, 32, 64, 1, 2, 128, 3, 0.35, 4},    // 27 8 waves, 144 KB
    // 28-32: wave-specialized (gemm_ws_kernel): WM x WN compute waves plus 4
    // DMA-only loader waves.  Measured on the packed C4 projections against
    // the best plan above: FFN2 (5430 x 1024 x 4096) 51 against 55.5 us,
    // out-proj 20.6 against 22.0 us, FFN1 59.7 against 60.2 us; QKV no gain.
    {kWs, 192, 128, 2, 2, 128, 4, 0.85, 1, 4},  // 28 wave tile 96x64, 160 KB
    {kWs, 192, 128, 2, 4, 128, 3, 0.85, 1, 4},  // 29 wave tile 96x32, 120 KB
    {kWs, 192, 128, 2, 4, 128, 4, 0.85, 1, 4},  // 30 wave tile 96x32, 160 KB
    {kWs, 192, 256, 2, 4, 128, 2, 0.85, 1, 4},  // 31 wave tile 96x64, 112 KB
    {kWs, 128, 256, 2, 4, 128, 3, 0.85, 1, 4},  // 32 wave tile 64x64, 144 KB
    // 33-35: panel rings (gemm_panel_kernel), 2 x 2 waves.
    {kPanel, 256, 256, 2, 2, 128, 2, 1.00},     // 33 wave tile 128x128, 128 KB
    {kPanel, 192, 128, 2, 2, 128, 2, 0.90},     // 34 wave tile 96x64, 80 KB, 2 WG/CU
    {kPanel, 128, 128, 2, 2, 128, 2, 0.90},     // 35 wave tile 64x64, 64 KB, 2 WG/CU
};
// fp32.
static const GemmPlan kPlans32[] = {
    {kStaged, 128, 128, 2, 2, 128, 2, 0.6},  // 0
    {kStaged, 64, 64, 2, 2, 128, 2, 0.4},    // 1
    {kDtl, 128, 128, 2, 2, 128, 2, 1.0},     // 2
    {kDtl, 256, 128, 2, 2, 128, 2, 1.0},     // 3
    {kDtl, 64, 64, 2, 2, 128, 2, 0.5},       // 4
    // 5: K split between four one-wave groups, for launches whose 64 x 64 tiles
    // leave most CUs idle (256 x 1024 x 1024 22.9 -> 9.4 us); 6: the tile
    // between 64 x 64 and 128 x 128 (5690 x 1024 x 1792 180 -> 168 us).
    {kDtl, 32, 32, 1, 1, 128, 2, 0.3, 4},    // 5 4 waves, 64 KB
    // (6's prior: never ahead of 2 in the fall-back)
    {kDtl, 128, 64, 2, 2, 128, 2, 0.5},      // 6 wave tile 64x32
};

template <typename T>
static const GemmPlan* plans(int* count) {
  if (sizeof(T) == 4) {
    *count = sizeof(kPlans32) / sizeof(kPlans32[0]);
    return kPlans32;
  }
  *count = sizeof(kPlans16) / sizeof(kPlans16[0]);
  return kPlans16;
}

struct GemmArgs {
  const void* a; int64_t lda; const void* w; int64_t ldw; const void* bias; void* c; int64_t ldc;
  int M, N, K; hipStream_t s;
  ResSrc src;  // kEpiResidualFrom's residual source (unused by the other epilogues)
};

// Launches plan `plan` of T's table with epilogue `epi` (the operands
// already checked against it).
template <typename T> int run_gemm(int plan, int epi, const GemmArgs& g);
extern template int run_gemm<float>(int, int, const GemmArgs&);
extern template int run_gemm<f16>(int, int, const GemmArgs&);
extern template int run_gemm<bf16>(int, int, const GemmArgs&);

}  // namespace tjk
