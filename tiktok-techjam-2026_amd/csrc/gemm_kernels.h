// MFMA GEMM with fused epilogues for the QKV, out-proj and FFN projections.
//
//   C[m, n] = epi( sum_k A[m, k] * W[n, k] + bias[n] )
//
// A is the [M, K] activation, W the nn.Linear [N, K] weight: both operands
// are K-contiguous, so both tiles are staged into LDS the same way and no
// transpose is needed anywhere.  This replaces torch.addmm at
// tjkernels/engine.py:245,247 and the addmm + gelu FFN fallback at
// tjkernels/kernels/__init__.py:88-89.
//
// Tiling (gfx950, wave64):
//   * a workgroup owns a BM x BN output tile; WM x WN waves each own a
//     (BM/WM) x (BN/WN) sub-tile made of 32x32 MFMA blocks;
//   * K advances in BK steps (64 for 2-byte types = 128 B per row, 32 for
//     fp32); each step's A and W tiles live in LDS with a 16-byte row pad
//     (row pitch 144 B), which makes the ds_read_b128 fragment reads of 16
//     consecutive rows bank-conflict free;
//   * LDS is double-buffered: global loads for step k+1 are issued into
//     registers before the MFMAs of step k and written to the other buffer
//     after them, one barrier per step;
//   * the MFMA's first operand is the W fragment and the second the A
//     fragment, so the accumulator holds C^T: every lane owns four
//     consecutive n of one output row m, which turns the epilogue into 8- or
//     16-byte row stores and lets bias/GELU/residual be applied per register;
//   * workgroups are renumbered so that each XCD (the hardware deals
//     workgroup i to XCD i % 8) walks a contiguous range of a GROUP_M-grouped
//     tile order, keeping the A rows and W columns it reuses in its own L2.
#pragma once

#include "gemm_plans.h"

namespace tjk {

template <typename T, int BM, int BN, int WM, int WN, int EPI>
__global__ __launch_bounds__(WM * WN * 64) void gemm_kernel(
    const T* __restrict__ A, int64_t lda, const T* __restrict__ W, int64_t ldw,
    const T* __restrict__ bias, void* __restrict__ Cv, int64_t ldc, int M, int N, int K, ResSrc src) {
  constexpr int NT = WM * WN * 64;
  constexpr int VEC = 16 / sizeof(T);            // elements per 16-byte chunk
  constexpr int BK = 128 / sizeof(T);            // 128 bytes of K per row
  constexpr int CPR = BK / VEC;                  // chunks per row (8)
  constexpr int LDK = BK + VEC;                  // padded LDS row pitch (elements)
  constexpr int KS = BK / 16;                    // 16-deep MFMA steps per BK
  constexpr int WTM = BM / WM, WTN = BN / WN;
  constexpr int FM = WTM / 32, FN = WTN / 32;
  constexpr int CA = BM * CPR / NT, CW = BN * CPR / NT;
  static_assert(CA * NT == BM * CPR && CW * NT == BN * CPR, "tile/thread mismatch");
  static_assert(FM >= 1 && FN >= 1, "wave tile too small");

  __shared__ __attribute__((aligned(16))) T smem[2][(BM + BN) * LDK];

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WN, wn = wave % WN;
  const int l32 = lane & 31, hi = lane >> 5;

  // ---- tile coordinates: XCD-contiguous ranges of a grouped order
  int pid_m, pid_n;
  tile_coords(blockIdx.x, (M + BM - 1) / BM, (N + BN - 1) / BN, pid_m, pid_n);
  const int m0 = pid_m * BM, n0 = pid_n * BN;

  // ---- global -> register staging
  uint4 ra[CA], rw[CW];
  auto load_tiles = [&](int k0) {
#pragma unroll
    for (int i = 0; i < CA; ++i) {
      const int c = tid + i * NT, row = c / CPR, kc = c % CPR;
      const int gm = m0 + row, gk = k0 + kc * VEC;
      ra[i] = (gm < M && gk < K) ? *reinterpret_cast<const uint4*>(A + (int64_t)gm * lda + gk)
                                 : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < CW; ++i) {
      const int c = tid + i * NT, row = c / CPR, kc = c % CPR;
      const int gn = n0 + row, gk = k0 + kc * VEC;
      rw[i] = (gn < N && gk < K) ? *reinterpret_cast<const uint4*>(W + (int64_t)gn * ldw + gk)
                                 : make_uint4(0, 0, 0, 0);
    }
  };
  auto store_tiles = [&](int buf) {
    T* sA = smem[buf];
    T* sW = smem[buf] + BM * LDK;
#pragma unroll
    for (int i = 0; i < CA; ++i) {
      const int c = tid + i * NT, row = c / CPR, kc = c % CPR;
      *reinterpret_cast<uint4*>(sA + row * LDK + kc * VEC) = ra[i];
    }
#pragma unroll
    for (int i = 0; i < CW; ++i) {
      const int c = tid + i * NT, row = c / CPR, kc = c % CPR;
      *reinterpret_cast<uint4*>(sW + row * LDK + kc * VEC) = rw[i];
    }
  };

  f32x16 acc[FN][FM];
#pragma unroll
  for (int i = 0; i < FN; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  const int nk = (K + BK - 1) / BK;
  load_tiles(0);
  store_tiles(0);
  __syncthreads();

  for (int kt = 0; kt < nk; ++kt) {
    const int cur = kt & 1;
    if (kt + 1 < nk) load_tiles((kt + 1) * BK);
    const T* sA = smem[cur] + (wm * WTM + l32) * LDK + hi * 8;
    const T* sW = smem[cur] + BM * LDK + (wn * WTN + l32) * LDK + hi * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      typename Mfma<T>::frag af[FM], wf[FN];
#pragma unroll
      for (int j = 0; j < FM; ++j) af[j] = Mfma<T>::load(sA + j * 32 * LDK + ks * 16);
#pragma unroll
      for (int i = 0; i < FN; ++i) wf[i] = Mfma<T>::load(sW + i * 32 * LDK + ks * 16);
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) Mfma<T>::mma(acc[i][j], wf[i], af[j]);
    }
    if (kt + 1 < nk) store_tiles(cur ^ 1);
    __syncthreads();
  }

  // The loop ends on a barrier, so the operand tiles are dead: reuse LDS.
  static_assert(NT / 64 * EpiStage<T, EPI, FN>::BYTES <= (int)sizeof(smem), "epilogue staging exceeds LDS");
  epilogue<T, EPI, FM, FN>(acc, bias, Cv, ldc, M, N, m0 + wm * WTM, n0 + wn * WTN, lane,
                           reinterpret_cast<char*>(&smem[0][0]) + wave * EpiStage<T, EPI, FN>::BYTES, NoPrefetch(),
                           nullptr, src);
}

template <typename T, int BM, int BN, int WM, int WN, int BKB, int STAGES, int EPI, int KSPLIT>
__global__ __launch_bounds__(WM * WN * KSPLIT * 64) void gemm_dtl_kernel(
    const T* __restrict__ A, int64_t lda, const T* __restrict__ W, int64_t ldw,
    const T* __restrict__ bias, void* __restrict__ Cv, int64_t ldc, int M, int N, int K, ResSrc src) {
  typedef DtlGeom<T, BM, BN, WM, WN, BKB, STAGES, KSPLIT> G;
  constexpr int NW = G::NW, FM = G::FM, FN = G::FN;
  __shared__ __attribute__((aligned(1024))) char smem[G::LDS];

  const int tid = threadIdx.x;
  const int lane = tid & 63, kg = (tid >> 6) / NW, wave = (tid >> 6) % NW;
  const int wm = wave / WN, wn = wave % WN;

  int pid_m, pid_n;
  tile_coords(blockIdx.x, (M + BM - 1) / BM, (N + BN - 1) / BN, pid_m, pid_n);
  const int m0 = pid_m * BM, n0 = pid_n * BN;

  // Bias and residual reads issued ahead of the operand DMAs, where their
  // registers fit beside the accumulators (plus ~144 for fragments and
  // addresses) without lowering the occupancy the LDS ring allows: their
  // round trip then overlaps the main loop instead of ending the launch,
  // which matters most for the short launches of a few hundred rows.  Wave
  // tiles above 4 blocks of 32 x 32 keep the bias loads in the epilogue and
  // prefetch only the residual, and only without a K split: there the
  // fragments already bring the wave close to its 256 architectural
  // registers (measured: 256 x 256 and 128 x 256 tiles spilled).
  constexpr int WG_PER_CU = 160 * 1024 / G::LDS;
  constexpr int WAVES_PER_SIMD = (WG_PER_CU * NW * KSPLIT + 3) / 4 > 1 ? (WG_PER_CU * NW * KSPLIT + 3) / 4 : 1;
  constexpr int BUDGET = 512 / WAVES_PER_SIMD - FM * FN * 16 - 144;
  constexpr int BIAS_REGS = FN * 4 * (int)sizeof(typename Quad<T>::raw) / 4;
  typedef ResPrefetch<FM, FN, T, EPI == kEpiResidualFrom> ResPre;
  constexpr int PRE_REGS = ResPre::REGS;
  constexpr bool SMALL = sizeof(T) == 2 && FM * FN <= 4;
  constexpr bool BIAS_PRE = SMALL && BIAS_REGS <= BUDGET;
  constexpr bool PREFETCH = epi_residual(EPI) && (KSPLIT == 1 || SMALL) &&
                            PRE_REGS + (BIAS_PRE ? BIAS_REGS : 0) <= BUDGET;
  typedef typename std::conditional<PREFETCH, ResPre, NoPrefetch>::type Pre;
  BiasRaw<T, FN> bpre;
  if constexpr (BIAS_PRE) bpre.load(bias, N, n0 + wn * G::WTN, lane);
  Pre pre;
  if constexpr (PREFETCH)
    pre.load(static_cast<const float*>(Cv), ldc, M, N, m0 + wm * G::WTM, n0 + wn * G::WTN, lane, src);

  f32x16 acc[FN][FM];
  zero_acc<T, FM, FN>(acc);
  dtl_accumulate<T, BM, BN, WM, WN, BKB, STAGES, KSPLIT>(smem, A, lda, W, ldw, M, N, K, m0, n0, acc);

  constexpr int ACCF = FN * FM * 16;                   // accumulator floats per lane
  constexpr int XCH = (KSPLIT - 1) * NW * ACCF * 64 * 4;  // exchange bytes
  static_assert(XCH + NW * EpiStage<T, EPI, FN>::BYTES <= G::LDS,
                "K-split exchange + epilogue staging exceed LDS");
  if constexpr (KSPLIT > 1) {
    // the groups' accumulators are summed (in group order) before the epilogue
    float* xch = reinterpret_cast<float*>(smem);
    if (kg > 0) {
      float* my = xch + (int64_t)((kg - 1) * NW + wave) * ACCF * 64;
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) my[((i * FM + j) * 16 + r) * 64 + lane] = acc[i][j][r];
    }
    __syncthreads();
    if (kg > 0) return;
#pragma unroll
    for (int p = 1; p < KSPLIT; ++p) {
      const float* ot = xch + (int64_t)((p - 1) * NW + wave) * ACCF * 64;
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[i][j][r] += ot[((i * FM + j) * 16 + r) * 64 + lane];
    }
  }
  // batched residual reads except in the register-tight tiles (K-split
  // groups, more than 8 accumulator blocks), where they spilled
  constexpr int RB = KSPLIT == 1 && FM * FN <= 8 ? kResBatch : 0;
  epilogue<T, EPI, FM, FN, Pre, RB>(acc, bias, Cv, ldc, M, N, m0 + wm * G::WTM, n0 + wn * G::WTN, lane,
                                    smem + XCH + wave * EpiStage<T, EPI, FN>::BYTES, pre,
                                    BIAS_PRE ? &bpre : nullptr, src);
}


// ---------------------------------------------------- wave-specialized GEMM
//
// The direct-to-LDS main loop above issues its DMA from the waves that run
// the MFMAs.  When the per-CU DMA rate saturates (measured on MI355X:
// ~35-44 B/clk per CU for buffer_load ... lds), a wave stalls at the issue
// of its next DMA instruction and, issuing in order, its MFMAs stall with
// it: the loop then takes about the DMA-only time plus the MFMA-only time
// (1.5x the larger of the two at the packed C4 shapes).  Here the two jobs
// go to different waves of the workgroup:
//   * NW = WM x WN compute waves read fragments from the ring and issue the
//     MFMAs (the same fragment reads, MFMA order and epilogue as
//     gemm_dtl_kernel, so the results are bitwise those of the class-1
//     plans);
//   * L loader waves only issue the LDS DMA of K tile kt + STAGES - 1 and
//     wait for tile kt + 1 to land.
// One barrier per K tile (B_kt, before the compute waves' last 16-deep step
// of tile kt) orders them: after B_kt tile kt + 1 has landed and tile kt's
// slot is free.  A final barrier ends the ring before the epilogue reuses
// its LDS; the loader waves then exit.
template <typename T, int BM, int BN, int WM, int WN, int STAGES, int L, int EPI>
__global__ __launch_bounds__((WM * WN + L) * 64) void gemm_ws_kernel(
    const T* __restrict__ A, int64_t lda, const T* __restrict__ W, int64_t ldw,
    const T* __restrict__ bias, void* __restrict__ Cv, int64_t ldc, int M, int N, int K, ResSrc src) {
  constexpr int BKB = 128;
  typedef DtlGeom<T, BM, BN, WM, WN, BKB, STAGES, 1> G;
  constexpr int NW = G::NW, KS = G::KS, CPS = G::CPS, WTM = G::WTM, WTN = G::WTN, FM = G::FM, FN = G::FN;
  constexpr int STAGE = G::STAGE;
  constexpr int NINST = (BM + BN) / G::RPI;  // 1 KB DMA instructions per K tile
  constexpr int NL = NINST / L;              // per loader wave
  static_assert(NINST % L == 0 && BM % G::RPI == 0, "DMA rows split over the loader waves");
  static_assert(STAGES >= 2 && (STAGES - 2) * NL <= 63, "vmcnt range");
  constexpr int STG = NW * EpiStage<T, EPI, FN>::BYTES;
  constexpr int LDS = STAGES * STAGE > STG ? STAGES * STAGE : STG;
  __shared__ __attribute__((aligned(1024))) char smem[LDS];

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  int pid_m, pid_n;
  tile_coords(blockIdx.x, (M + BM - 1) / BM, (N + BN - 1) / BN, pid_m, pid_n);
  const int m0 = pid_m * BM, n0 = pid_n * BN;
  const int nk = (K + G::BK - 1) / G::BK;

  if (wave >= NW) {
    // ------------------------------------------------------------ loaders
    const int lw = wave - NW;
    const int64_t a_rows = min((int64_t)BM, (int64_t)(M - m0));
    const int64_t w_rows = min((int64_t)BN, (int64_t)(N - n0));
    const __amdgpu_buffer_rsrc_t rsa = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(A + (int64_t)m0 * lda), (short)0, (int)(a_rows * lda * (int64_t)sizeof(T)), 0x00020000);
    const __amdgpu_buffer_rsrc_t rsw = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(W + (int64_t)n0 * ldw), (short)0, (int)(w_rows * ldw * (int64_t)sizeof(T)), 0x00020000);
    // instruction q of loader lw fills rows (q L + lw) RPI .. +RPI-1 of the
    // stacked (A; W) tile; lane l lands at byte 16 l: row + l / CPR,
    // physical chunk l % CPR, so it fetches logical chunk (l % CPR) ^ swz(row)
    // (the pieces of a last K tile past K point outside the range: zeros; L is
    // even, so every instruction of a lane fetches the same chunk of its row)
    static_assert(L % 2 == 0 && (BM / G::RPI) % 2 == 0, "row parity of the DMA instructions");
    const uint32_t kend = (uint32_t)K * (uint32_t)sizeof(T);
    const uint32_t lcb = (uint32_t)(((lane % G::CPR) ^ swz<BKB>(lw * G::RPI + lane / G::CPR)) << 4);
    auto dma = [&](int t, int q) {
      char* sb = smem + (t % STAGES) * STAGE;
      const int base = (q * L + lw) * G::RPI;  // wave-uniform
      const uint32_t kb = (uint32_t)(t * BKB) + lcb < kend ? (uint32_t)(t * BKB) : kPastEnd;
      if (base < BM) {
        const int r = base + lane / G::CPR;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rsa, (lds_void*)(sb + base * BKB), 16,
            (uint32_t)(r * lda * (int64_t)sizeof(T)) + (uint32_t)(((lane % G::CPR) ^ swz<BKB>(r)) << 4) + kb, 0, 0, 0);
      } else {
        const int r = base - BM + lane / G::CPR;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rsw, (lds_void*)(sb + base * BKB), 16,
            (uint32_t)(r * ldw * (int64_t)sizeof(T)) + (uint32_t)(((lane % G::CPR) ^ swz<BKB>(r)) << 4) + kb, 0, 0, 0);
      }
    };
    for (int t = 0; t < STAGES - 1 && t < nk; ++t) {
#pragma unroll
      for (int q = 0; q < NL; ++q) dma(t, q);
    }
    // tile 0 landed (the tiles issued after it may still be in flight)
    if (nk >= STAGES - 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((STAGES - 2) * NL) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();  // B_-1
    for (int k = 0; k < nk; ++k) {
      // tile k + STAGES - 1 into the slot tile k - 1 freed at B_{k-1};
      // then tile k + 1 landed before B_k
      const int t = k + STAGES - 1;
      if (t < nk) {
#pragma unroll
        for (int q = 0; q < NL; ++q) dma(t, q);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((STAGES - 2) * NL) : "memory");
      } else {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      __builtin_amdgcn_s_barrier();  // B_k
    }
    __builtin_amdgcn_s_barrier();  // B_final
    return;
  }

  // ------------------------------------------------------------- compute
  const int wm = wave / WN, wn = wave % WN;
  const int l32 = lane & 31, hi = lane >> 5;
  // The epilogue's bias and residual reads go out before the main loop where
  // the registers allow (accumulators, two fragment sets and address
  // registers counted against the per-wave share of the register file):
  // their round trip then overlaps the main loop.
  constexpr int WPS = (NW + L + 3) / 4;  // waves per SIMD (one workgroup per CU)
  constexpr int AVAIL = (512 / WPS) & ~7;
  // (the residual first: its read-modify-write is most of a residual
  // epilogue; 36 overhead registers, 44 with a ring whose slot count is not
  // a power of two, keeps every plan here free of spills)
  constexpr int USED = FM * FN * 16 + 2 * (FM + FN) * 4 + ((STAGES & (STAGES - 1)) ? 44 : 36);
  constexpr int BIAS_REGS = FN * 4 * (int)sizeof(typename Quad<T>::raw) / 4;
  typedef ResPrefetch<FM, FN, T, EPI == kEpiResidualFrom> ResPre;
  constexpr int PRE_REGS = ResPre::REGS;
  constexpr bool PREFETCH = epi_residual(EPI) && USED + PRE_REGS <= AVAIL;
  constexpr bool BIAS_PRE = USED + BIAS_REGS + (PREFETCH ? PRE_REGS : 0) <= AVAIL;
  typedef typename std::conditional<PREFETCH, ResPre, NoPrefetch>::type Pre;
  BiasRaw<T, FN> bpre;
  if constexpr (BIAS_PRE) bpre.load(bias, N, n0 + wn * WTN, lane);
  Pre pre;
  if constexpr (PREFETCH)
    pre.load(static_cast<const float*>(Cv), ldc, M, N, m0 + wm * WTM, n0 + wn * WTN, lane, src);
  const int sw = swz<BKB>(l32);
  typedef typename Mfma<T>::frag Frag;
  auto frag_at = [&](const char* rowbase, int ks) -> Frag {
    return *reinterpret_cast<const Frag*>(rowbase + (((CPS * ks + hi) ^ sw) << 4));
  };
  f32x16 acc[FN][FM];
  zero_acc<T, FM, FN>(acc);
  constexpr int NMF = FN * FM, NDS = FN + FM;
  constexpr int NSLOT = NMF > NDS ? NMF : NDS;
  Frag fa[2][FM], fw[2][FN];
  __builtin_amdgcn_s_barrier();  // B_-1: tile 0 landed
  __builtin_amdgcn_sched_barrier(0);
  {
    const char* sa = smem + (wm * WTM + l32) * BKB;
    const char* sw_ = smem + BM * BKB + (wn * WTN + l32) * BKB;
#pragma unroll
    for (int j = 0; j < FM; ++j) fa[0][j] = frag_at(sa + j * 32 * BKB, 0);
#pragma unroll
    for (int i = 0; i < FN; ++i) fw[0][i] = frag_at(sw_ + i * 32 * BKB, 0);
  }
  // Same schedule as dtl_accumulate: MFMA m of a step, then fragment read m
  // of the next step; the barrier precedes the last step of a tile, whose
  // fragments are in registers, and the next tile's first fragments are
  // read during the last step's MFMAs.  (The slot after the last tile is
  // read too; those fragments are never used.)
  for (int kt = 0; kt < nk; ++kt) {
    const char* st = smem + (kt % STAGES) * STAGE;
    const char* sa = st + (wm * WTM + l32) * BKB;
    const char* sw_ = st + BM * BKB + (wn * WTN + l32) * BKB;
    const char* nx = smem + ((kt + 1) % STAGES) * STAGE;
    const char* na = nx + (wm * WTM + l32) * BKB;
    const char* nw = nx + BM * BKB + (wn * WTN + l32) * BKB;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int b = ks & 1;
      const bool last = ks + 1 == KS;
      const char* ra = last ? na : sa;
      const char* rw = last ? nw : sw_;
      const int rks = last ? 0 : ks + 1;
      if (last) {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // my reads of slot kt are done
        __builtin_amdgcn_s_barrier();                        // B_kt
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int m = 0; m < NSLOT; ++m) {
        if (m < NMF) Mfma<T>::mma(acc[m / FM][m % FM], fw[b][m / FM], fa[b][m % FM]);
        if (m < FM) fa[b ^ 1][m] = frag_at(ra + m * 32 * BKB, rks);
        else if (m < NDS) fw[b ^ 1][m - FM] = frag_at(rw + (m - FM) * 32 * BKB, rks);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();  // B_final: every ring read done, every DMA landed
  // (the tiles that cannot take the prefetch are register-tight: their
  // residual pieces are read one by one, which spills nothing)
  epilogue<T, EPI, FM, FN, Pre, 0>(acc, bias, Cv, ldc, M, N, m0 + wm * WTM, n0 + wn * WTN, lane,
                                   smem + wave * EpiStage<T, EPI, FN>::BYTES, pre, BIAS_PRE ? &bpre : nullptr,
                                   src);
}

// ------------------------------------------------------- panel-ring GEMM
//
// panel_accumulate's main loop (gemm_tiles.h) under the shared epilogue: four
// waves, wave tile (32 FM) x (32 FN).  The same K order as the class-1 plans:
// a 16x16x32 MFMA gives the bits of two 32x32x16 ones (tests compare every
// plan of the class).  256 x 256 fills a CU (128 KB of LDS, 256 AGPRs, nothing in
// scratch); the smaller tiles run two workgroups per CU, whose main loops cover
// each other's prologue and epilogue.  Measured (bf16, one box, against the best
// other plan): 8192^3 825 -> 715 us (plan 8), 8192 x 2048 x 8192 with the
// residual 219 -> 190 us (8), 5430 x 4096 x 1024 with GELU 53.0 -> 50.1 us (192 x
// 128 tiles; plan 31).  192 x 256, 256 x 128 and 192 x 192 tiles of this
// kernel were no faster than these on any shape tried.
template <typename T, int FM, int FN, int EPI>
__global__ __launch_bounds__(256, (PanelGeom<FM, FN>::LDS <= 80 * 1024 ? 2 : 1)) void gemm_panel_kernel(
    const T* __restrict__ A, int64_t lda, const T* __restrict__ W, int64_t ldw,
    const T* __restrict__ bias, void* __restrict__ Cv, int64_t ldc, int M, int N, int K, ResSrc src) {
  typedef PanelGeom<FM, FN> G;
  static_assert(4 * EpiStage<T, EPI, FN>::BYTES <= G::LDS, "epilogue staging exceeds LDS");
  __shared__ __attribute__((aligned(1024))) char smem[G::LDS];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int pid_m, pid_n;
  tile_coords(blockIdx.x, (M + G::BM - 1) / G::BM, (N + G::BN - 1) / G::BN, pid_m, pid_n);
  const int m0 = pid_m * G::BM, n0 = pid_n * G::BN;
  const int mw = m0 + (wave >> 1) * 32 * FM, nw = n0 + (wave & 1) * 32 * FN;

  // Bias and residual reads ahead of the main loop where they fit beside the
  // accumulators, the fragments of a K tile and ~40 other registers.
  constexpr int BUDGET = (G::LDS <= 80 * 1024 ? 256 : 512) - FM * FN * 16 - (FM + FN) * 16 - 40;
  constexpr int BIAS_REGS = FN * 2 * (int)sizeof(typename Quad<T>::raw) / 4;
  typedef ResPrefetch<FM, FN, T, EPI == kEpiResidualFrom> ResPre;
  constexpr bool BIAS_PRE = BIAS_REGS <= BUDGET && FM * FN <= 8;
  constexpr bool PREFETCH = epi_residual(EPI) && ResPre::REGS + BIAS_REGS <= BUDGET;
  typedef typename std::conditional<PREFETCH, ResPre, NoPrefetch>::type Pre;
  BiasRaw<T, FN, true> bpre;
  if constexpr (BIAS_PRE) bpre.load(bias, N, nw, lane);
  Pre pre;
  if constexpr (PREFETCH) pre.load(static_cast<const float*>(Cv), ldc, M, N, mw, nw, lane, src);

  Acc16<FM, FN> acc;
#pragma unroll
  for (int i = 0; i < 2 * FN; ++i)
#pragma unroll
    for (int j = 0; j < 2 * FM; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  panel_accumulate<T, FM, FN>(smem, A, lda, W, ldw, M, N, K, m0, n0, acc);
  epilogue<T, EPI, FM, FN, Pre, kResBatch, true>(acc, bias, Cv, ldc, M, N, mw, nw, lane,
                                                 smem + wave * EpiStage<T, EPI, FN>::BYTES, pre,
                                                 BIAS_PRE ? &bpre : nullptr, src);
}

// Kernel selection by plan kind through a specialised struct (the host stub
// of a kernel launched under `if constexpr` is not always emitted).
template <int KIND> struct Launcher;
template <> struct Launcher<kStaged> {
  template <typename T, int BM, int BN, int WM, int WN, int EPI>
  static int go(const GemmArgs& g) {
    const dim3 grid(((g.M + BM - 1) / BM) * ((g.N + BN - 1) / BN));
    hipLaunchKernelGGL((gemm_kernel<T, BM, BN, WM, WN, EPI>), grid, dim3(WM * WN * 64), 0, g.s, (const T*)g.a,
                       g.lda, (const T*)g.w, g.ldw, (const T*)g.bias, g.c, g.ldc, g.M, g.N, g.K, g.src);
    return TJK_OK;
  }
};
template <int BKB, int STAGES, int KSPLIT = 1> struct DtlLauncher {
  template <typename T, int BM, int BN, int WM, int WN, int EPI>
  static int go(const GemmArgs& g) {
    const dim3 grid(((g.M + BM - 1) / BM) * ((g.N + BN - 1) / BN));
    hipLaunchKernelGGL((gemm_dtl_kernel<T, BM, BN, WM, WN, BKB, STAGES, EPI, KSPLIT>), grid,
                       dim3(WM * WN * KSPLIT * 64), 0, g.s, (const T*)g.a, g.lda, (const T*)g.w, g.ldw,
                       (const T*)g.bias, g.c, g.ldc, g.M, g.N, g.K, g.src);
    return TJK_OK;
  }
};

template <typename L, typename T, int BM, int BN, int WM, int WN>
static int launch_epi(int epi, const GemmArgs& g) {
  switch (epi) {
    case TJK_EPI_BIAS: return L::template go<T, BM, BN, WM, WN, TJK_EPI_BIAS>(g);
    case TJK_EPI_BIAS_GELU: return L::template go<T, BM, BN, WM, WN, TJK_EPI_BIAS_GELU>(g);
    case kEpiResidualFrom: return L::template go<T, BM, BN, WM, WN, kEpiResidualFrom>(g);
    default: return L::template go<T, BM, BN, WM, WN, TJK_EPI_BIAS_RESIDUAL>(g);
  }
}

template <int STAGES, int L> struct WsLauncher {
  template <typename T, int BM, int BN, int WM, int WN, int EPI>
  static int go(const GemmArgs& g) {
    const dim3 grid(((g.M + BM - 1) / BM) * ((g.N + BN - 1) / BN));
    hipLaunchKernelGGL((gemm_ws_kernel<T, BM, BN, WM, WN, STAGES, L, EPI>), grid, dim3((WM * WN + L) * 64), 0,
                       g.s, (const T*)g.a, g.lda, (const T*)g.w, g.ldw, (const T*)g.bias, g.c, g.ldc, g.M, g.N,
                       g.K, g.src);
    return TJK_OK;
  }
};

struct PanelLauncher {
  template <typename T, int BM, int BN, int WM, int WN, int EPI>
  static int go(const GemmArgs& g) {
    static_assert(WM == 2 && WN == 2, "four waves");
    const dim3 grid(((g.M + BM - 1) / BM) * ((g.N + BN - 1) / BN));
    hipLaunchKernelGGL((gemm_panel_kernel<T, BM / 64, BN / 64, EPI>), grid, dim3(256), 0, g.s, (const T*)g.a, g.lda,
                       (const T*)g.w, g.ldw, (const T*)g.bias, g.c, g.ldc, g.M, g.N, g.K, g.src);
    return TJK_OK;
  }
};

typedef Launcher<kStaged> St;
typedef DtlLauncher<128, 2> D2;
typedef DtlLauncher<128, 2, 2> D2K2;
typedef DtlLauncher<128, 2, 4> D2K4;
typedef DtlLauncher<128, 4, 2> D4K2;
typedef DtlLauncher<128, 3, 2> D3K2;
typedef DtlLauncher<128, 4, 4> D4K4;
typedef DtlLauncher<128, 3, 4> D3K4;
typedef DtlLauncher<128, 4> D4;
typedef DtlLauncher<128, 6> D6;
typedef DtlLauncher<128, 8> D8;
typedef WsLauncher<4, 4> W4;
typedef WsLauncher<3, 4> W3;
typedef WsLauncher<2, 4> W2;

template <typename T>
int run_gemm(int plan, int epi, const GemmArgs& g) {
  int rc = TJK_OK;
#define TJK_GEMM_CASE(ID, L, BM, BN, WM, WN) \
  case ID: rc = launch_epi<L, T, BM, BN, WM, WN>(epi, g); break;
  if constexpr (sizeof(T) == 4) {
    switch (plan) {
      TJK_GEMM_CASE(0, St, 128, 128, 2, 2)
      TJK_GEMM_CASE(1, St, 64, 64, 2, 2)
      TJK_GEMM_CASE(2, D2, 128, 128, 2, 2)
      TJK_GEMM_CASE(3, D2, 256, 128, 2, 2)
      TJK_GEMM_CASE(4, D2, 64, 64, 2, 2)
      TJK_GEMM_CASE(5, D2K4, 32, 32, 1, 1)
      TJK_GEMM_CASE(6, D2, 128, 64, 2, 2)
    }
  } else {
    switch (plan) {
      TJK_GEMM_CASE(0, St, 256, 256, 2, 2)
      TJK_GEMM_CASE(1, St, 256, 128, 2, 2)
      TJK_GEMM_CASE(2, St, 128, 256, 2, 2)
      TJK_GEMM_CASE(3, St, 128, 128, 2, 2)
      TJK_GEMM_CASE(4, St, 64, 64, 2, 2)
      TJK_GEMM_CASE(5, St, 256, 256, 2, 4)
      TJK_GEMM_CASE(6, D2, 256, 256, 2, 2)
      TJK_GEMM_CASE(7, D2, 128, 128, 2, 2)
      TJK_GEMM_CASE(8, D2, 256, 256, 2, 4)
      TJK_GEMM_CASE(9, D2, 64, 64, 2, 2)
      TJK_GEMM_CASE(10, D2, 256, 128, 2, 2)
      TJK_GEMM_CASE(11, D2, 128, 256, 2, 2)
      TJK_GEMM_CASE(12, D2, 192, 128, 2, 2)
      TJK_GEMM_CASE(13, D2, 192, 256, 2, 4)
      TJK_GEMM_CASE(14, D2, 192, 384, 2, 4)
      TJK_GEMM_CASE(15, D2, 96, 128, 1, 4)
      TJK_GEMM_CASE(16, D2K2, 192, 128, 2, 2)
      TJK_GEMM_CASE(17, D2K2, 128, 128, 2, 2)
      TJK_GEMM_CASE(18, D4, 192, 128, 2, 2)
      TJK_GEMM_CASE(19, D8, 64, 64, 2, 2)
      TJK_GEMM_CASE(20, D6, 128, 64, 2, 2)
      TJK_GEMM_CASE(21, D2K4, 64, 64, 2, 2)
      TJK_GEMM_CASE(22, D4K2, 64, 64, 2, 2)
      TJK_GEMM_CASE(23, D3K2, 128, 64, 2, 2)
      TJK_GEMM_CASE(24, D4K2, 32, 64, 1, 2)
      TJK_GEMM_CASE(25, D4K2, 32, 32, 1, 1)
      TJK_GEMM_CASE(26, D4K4, 32, 32, 1, 1)
      TJK_GEMM_CASE(27, D3K4, 32, 64, 1, 2)
      TJK_GEMM_CASE(28, W4, 192, 128, 2, 2)
      TJK_GEMM_CASE(29, W3, 192, 128, 2, 4)
      TJK_GEMM_CASE(30, W4, 192, 128, 2, 4)
      TJK_GEMM_CASE(31, W2, 192, 256, 2, 4)
      TJK_GEMM_CASE(32, W3, 128, 256, 2, 4)
      TJK_GEMM_CASE(33, PanelLauncher, 256, 256, 2, 2)
      TJK_GEMM_CASE(34, PanelLauncher, 192, 128, 2, 2)
      TJK_GEMM_CASE(35, PanelLauncher, 128, 128, 2, 2)
    }
  }
#undef TJK_GEMM_CASE
  if (rc != TJK_OK) return rc;
  return check_launch("tjk_gemm_bias");
}

}  // namespace tjk
