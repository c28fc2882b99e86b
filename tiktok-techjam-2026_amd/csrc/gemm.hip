// Entry points of the GEMM (tjk_gemm_bias, tjk_gemm_bias_residual_from):
// argument checks and the default tile choice.  The kernels are in
// gemm_kernels.h, compiled once per element type.

#include "gemm_plans.h"

namespace tjk {

static bool dtl_ok(const GemmPlan& p, int64_t k, int64_t lda, int64_t ldw, int es) {
  return k % (p.bkb / es) == 0 && (lda * es) % 16 == 0 && (ldw * es) % 16 == 0;
}

// K-summation class of the default tile (plans of a class give the same
// bits), by the shape alone; M counts in buckets of 64 rows, as the tile
// timing of tjkernels/tiles.py (k_class) keys its shapes, so that a timed and
// a default choice always agree in class.
template <typename T>
static int k_class(int64_t M, int64_t N, int64_t K) {
  const int64_t m = (M + 63) / 64 * 64;
  if (sizeof(T) == 4) {
    // at 128 tiles of 64 x 64 the split is 1.2-1.8 times as fast, at 192 with
    // K >= 2048 1.2; at 192 with less K, and at 256, it is slower
    const int64_t tiles = m / 64 * ((N + 63) / 64);
    return (tiles <= 128 && K >= 256) || (tiles <= 192 && K >= 2048) ? 4 : 1;
  }
  if ((m + 31) / 32 * ((N + 63) / 64) <= 256 && K >= 2048) return 4;
  // Two K groups while 128 x 64 tiles are at most one per CU; with K < 768 and
  // more than half of the CUs at work, wide outputs (few rows of tiles to share
  // W between) are faster unsplit: 700 x 2048 x 512 7.3 -> 6.8 us, 1024 x 1536 x
  // 512 7.3 -> 6.9; at N = 512 4096 x 512 x 512 into the fp32 residual is not
  // (7.8 -> 8.1).
  const int64_t tiles = (m + 127) / 128 * ((N + 63) / 64);
  return tiles <= 256 && K >= 512 && (K >= 768 || N < 1024 || tiles <= 128) ? 2 : 1;
}

// Estimated microseconds of a launch on MI355X: with `tiles`
// workgroups, `per_cu` of them resident per CU, a launch is `rounds` fillings
// of the chip, in which the fullest CU runs `load` workgroups in all, each of
// `steps` K tiles (per K group; the panel ring runs an even number), and stores
// `mb` MB of output (read and written, for a residual):
//   c0 + c1 rounds + c2 rounds steps + c3 load + c4 load steps + c5 mb
// (mb at 5 TB/s).  The coefficients are a non-negative least squares fit by
// relative error to launches timed with every plan; profiles/gemm_tiles.csv
// holds the launches and gemm_tiles.md what the estimate loses on them.  One K
// group: 2013 launches (16 to 16384 rows, widths and K up to 8192, every
// epilogue), weighted towards plans near the best of their launch; the tile
// picked is 0.3% slower than the best of the eight (geometric mean), and 9%
// faster than the fixed rule before it (8 from 512 tiles of 256 x 256, 7 from
// 128 of 128 x 128, else 9), 7 launches more than 2% slower, none 5%.  Without
// 7, 8 and the panel ring's even steps it was 0.9% slower than the best and 32
// launches more than 5% slower than that rule, most with K <= 384 and a
// residual.  Two and four K groups: the best tile but for 4 of 1547 launches.
// fp32: 0.5% slower than the best tile over 336 launches, none slower than the
// rule before it (rounds x area / prior); K split in four, 364 launches, always
// faster than any unsplit tile.
struct AutoTile {
  int plan, per_cu;
  float c[6];
};
static const AutoTile kAuto16[] = {
    // one K group: 64 x 64, 96 x 128, panels 192 x 128, 128 x 128 and 256 x 256,
    // 192 x 384, 128 x 128, 256 x 256
    {9, 5, {1.954f, 0.733f, 0.089f, 0.411f, 0.163f, 0.362f}},
    {15, 2, {0.980f, 1.220f, 0.379f, 1.098f, 0.185f, 0.442f}},
    {34, 2, {1.536f, 2.753f, 0.131f, 0.924f, 0.505f, 0.498f}},
    {35, 2, {1.513f, 2.455f, 0.129f, 0.170f, 0.347f, 0.652f}},
    {33, 1, {0.000f, 0.000f, 1.323f, 8.871f, 0.000f, 0.575f}},
    {14, 1, {0.000f, 0.000f, 1.638f, 7.071f, 0.000f, 0.726f}},
    {7, 2, {1.595f, 1.016f, 0.289f, 1.104f, 0.318f, 0.529f}},
    {8, 1, {0.000f, 0.000f, 1.499f, 5.760f, 0.000f, 0.625f}},
    // two K groups: 32 x 32, 32 x 64, 64 x 64, 128 x 64
    {25, 2, {1.108f, 1.764f, 0.151f, 0.325f, 0.073f, 0.000f}},
    {24, 1, {0.846f, 2.472f, 0.000f, 0.000f, 0.261f, 0.000f}},
    {22, 1, {0.627f, 2.796f, 0.322f, 0.000f, 0.000f, 0.390f}},
    {23, 1, {0.190f, 3.885f, 0.493f, 0.000f, 0.000f, 0.629f}},
    // four K groups: 32 x 32, 32 x 64
    {26, 1, {0.897f, 2.638f, 0.308f, 0.000f, 0.000f, 0.000f}},
    {27, 1, {0.580f, 3.114f, 0.000f, 0.000f, 0.464f, 0.091f}},
};

static const AutoTile kAuto32[] = {
    // 128 x 128, 64 x 64, 128 x 64; the one tile with four K groups
    {2, 2, {3.105f, 0.670f, 0.234f, 1.139f, 1.709f, 0.626f}},
    {4, 5, {2.625f, 0.000f, 0.169f, 0.000f, 0.469f, 1.167f}},
    {6, 3, {3.423f, 0.000f, 0.204f, 0.000f, 0.874f, 1.150f}},
    {5, 2, {}},
};

static bool span_ok(const GemmPlan& p, int64_t lda, int64_t ldw, int es) {
  return p.kind == kStaged || ((int64_t)p.bm * lda * es <= INT32_MAX && (int64_t)p.bn * ldw * es <= INT32_MAX);
}

// The tile of `table` with the least estimate in the shape's K class, or -1.
template <typename T, int NT>
static int least_estimate(const AutoTile (&table)[NT], const GemmPlan* p, int64_t M, int64_t N, int64_t K, int64_t lda,
                          int64_t ldw, int epi) {
  constexpr int BK = 128 / sizeof(T);
  const int cls = k_class<T>(M, N, K);
  const float mb = (float)M * (float)N * (epi_residual(epi) ? 8.f : (float)sizeof(T)) / 5e6f;
  const int64_t ktiles = (K + BK - 1) / BK;
  int best = -1;
  float best_us = 0.f;
  for (const AutoTile& t : table) {
    const GemmPlan& q = p[t.plan];
    if (q.ksplit != cls || !span_ok(q, lda, ldw, sizeof(T))) continue;
    const int64_t tiles = ((M + q.bm - 1) / q.bm) * ((N + q.bn - 1) / q.bn), slots = 256 * t.per_cu;
    const int64_t full = tiles / slots, rest = tiles % slots;
    const float rounds = (float)(full + (rest > 0)), load = (float)(full * t.per_cu + (rest + 255) / 256);
    const float steps = (float)(q.kind == kPanel ? ktiles + (ktiles & 1) : ktiles) / (float)cls;
    const float us = t.c[0] + rounds * (t.c[1] + t.c[2] * steps) + load * (t.c[3] + t.c[4] * steps) + t.c[5] * mb;
    if (best < 0 || us < best_us) {
      best = t.plan;
      best_us = us;
    }
  }
  return best;
}

// Default tile choice: the least estimate.  The direct-to-LDS kernels take
// any K here: pieces of the last K tile past K arrive as zeros.  (A plan asked
// for by id takes whole K tiles only.)  Rows too far apart for those tiles'
// 31-bit offsets go by the least (full-chip rounds of 256 workgroups) x (tile
// area / prior) over the plans with one K group that take the K: staged, or
// refused; fp32 ones of class 4 take its tile as far as 64 x 64 tiles reach.
template <typename T>
static int auto_plan(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldw, int epi) {
  int count;
  const GemmPlan* p = plans<T>(&count);
  if constexpr (sizeof(T) == 2) {
    const int narrow = ((M + 127) / 128) * ((N + 127) / 128) >= 128 ? 7 : 9;
    if (K % 64 == 0 && !span_ok(p[narrow], lda, ldw, sizeof(T))) return narrow;
    const int best = least_estimate<T>(kAuto16, p, M, N, K, lda, ldw, epi);
    if (best >= 0) return best;
  } else {
    if (span_ok(p[3], lda, ldw, sizeof(T))) return least_estimate<T>(kAuto32, p, M, N, K, lda, ldw, epi);
    if (k_class<T>(M, N, K) == 4 && span_ok(p[4], lda, ldw, sizeof(T))) return 5;
  }
  int best = 0;
  double best_cost = 1e300;
  for (int i = 0; i < count; ++i) {
    if (p[i].ksplit > 1 || (p[i].kind != kStaged && !dtl_ok(p[i], K, lda, ldw, sizeof(T)))) continue;
    const int64_t tiles = ((M + p[i].bm - 1) / p[i].bm) * ((N + p[i].bn - 1) / p[i].bn);
    const int64_t rounds = (tiles + 255) / 256;
    const double cost = (double)rounds * p[i].bm * p[i].bn / p[i].eff;
    if (cost < best_cost * 0.999) {
      best_cost = cost;
      best = i;
    }
  }
  return best;
}

template <typename T>
static int gemm_checked(const void* a, int64_t lda, const void* w, int64_t ldw, const void* bias, void* c,
                        int64_t ldc, int64_t m, int64_t n, int64_t k, int epi, int plan, hipStream_t s,
                        const ResSrc& src = ResSrc{nullptr, 0, nullptr, 0, nullptr}) {
  int count;
  const GemmPlan* p = plans<T>(&count);
  if (plan < -1 || plan >= count) return fail(TJK_EINVAL, "tjk_gemm_bias: plan %d out of range [-1,%d)", plan, count);
  const bool by_rule = plan == -1;
  if (by_rule) plan = auto_plan<T>(m, n, k, lda, ldw, epi);
  if (!by_rule && p[plan].kind != kStaged && !dtl_ok(p[plan], k, lda, ldw, sizeof(T)))
    return fail(TJK_EUNSUPPORTED, "tjk_gemm_bias: plan %d needs k %% %d == 0", plan, (int)(p[plan].bkb / sizeof(T)));
  if (!span_ok(p[plan], lda, ldw, sizeof(T)))
    return fail(TJK_EUNSUPPORTED, "tjk_gemm_bias: leading dimension too large for plan %d", plan);
  const GemmArgs g{a, lda, w, ldw, bias, c, ldc, (int)m, (int)n, (int)k, s, src};
  return run_gemm<T>(plan, epi, g);
}

}  // namespace tjk

using namespace tjk;

extern "C" int tjk_gemm_plan_count(int dtype) {
  int count = 0;
  if (dtype == TJK_F32) plans<float>(&count);
  else if (dtype == TJK_F16 || dtype == TJK_BF16) plans<bf16>(&count);
  else return fail(TJK_EINVAL, "tjk_gemm_plan_count: bad dtype %d", dtype);
  return count;
}

extern "C" int tjk_gemm_plan_info(int dtype, int id, int* block_m, int* block_n, int* waves, int* k_groups) {
  int count = 0;
  const GemmPlan* p;
  if (dtype == TJK_F32) p = plans<float>(&count);
  else if (dtype == TJK_F16 || dtype == TJK_BF16) p = plans<bf16>(&count);
  else return fail(TJK_EINVAL, "tjk_gemm_plan_info: bad dtype %d", dtype);
  if (id < 0 || id >= count) return fail(TJK_EINVAL, "tjk_gemm_plan_info: plan %d out of range", id);
  if (block_m) *block_m = p[id].bm;
  if (block_n) *block_n = p[id].bn;
  if (waves) *waves = p[id].wm * p[id].wn * p[id].ksplit + p[id].loaders;
  if (k_groups) *k_groups = p[id].ksplit;
  return TJK_OK;
}

extern "C" int tjk_gemm_default_plan(int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldw, int dtype,
                                     int epilogue) {
  if (m <= 0 || n <= 0 || k < 0 || lda < k || ldw < k || m > INT32_MAX || n > INT32_MAX || k > INT32_MAX)
    return fail(TJK_EINVAL, "tjk_gemm_default_plan: bad shape");
  if (epilogue < TJK_EPI_BIAS || epilogue > TJK_EPI_BIAS_RESIDUAL)
    return fail(TJK_EINVAL, "tjk_gemm_default_plan: bad epilogue %d", epilogue);
  if (dtype == TJK_F32) return auto_plan<float>(m, n, k, lda, ldw, epilogue);
  if (dtype == TJK_F16 || dtype == TJK_BF16) return auto_plan<bf16>(m, n, k, lda, ldw, epilogue);
  return fail(TJK_EINVAL, "tjk_gemm_default_plan: bad dtype %d", dtype);
}

extern "C" int tjk_gemm_bias(const void* a, int64_t lda, const void* w, int64_t ldw,
                             const void* bias, void* c, int64_t ldc,
                             int64_t m, int64_t n, int64_t k,
                             int dtype, int epilogue, int plan_id, void* stream) {
  if (m < 0 || n < 0 || k < 0) return fail(TJK_EINVAL, "tjk_gemm_bias: negative shape");
  if (m == 0 || n == 0) return TJK_OK;
  if (!a || !w || !c) return fail(TJK_EINVAL, "tjk_gemm_bias: null pointer");
  if (m > INT32_MAX || n > INT32_MAX || k > INT32_MAX) return fail(TJK_EUNSUPPORTED, "tjk_gemm_bias: shape exceeds int32");
  if (epilogue < TJK_EPI_BIAS || epilogue > TJK_EPI_BIAS_RESIDUAL)
    return fail(TJK_EINVAL, "tjk_gemm_bias: bad epilogue %d", epilogue);
  if (dtype != TJK_F32 && dtype != TJK_F16 && dtype != TJK_BF16) return fail(TJK_EINVAL, "tjk_gemm_bias: bad dtype %d", dtype);
  const int es = dtype_size(dtype), vec = 16 / es;
  if (k % vec) return fail(TJK_EUNSUPPORTED, "tjk_gemm_bias: k=%lld must be a multiple of %d", (long long)k, vec);
  if (n % 4) return fail(TJK_EUNSUPPORTED, "tjk_gemm_bias: n=%lld must be a multiple of 4", (long long)n);
  if (lda < k || ldw < k || ldc < n) return fail(TJK_EINVAL, "tjk_gemm_bias: leading dimension too small");
  if (lda % vec || ldw % vec) return fail(TJK_EUNSUPPORTED, "tjk_gemm_bias: lda/ldw must be multiples of %d", vec);
  if (ldc % 4) return fail(TJK_EUNSUPPORTED, "tjk_gemm_bias: ldc must be a multiple of 4");
  const int cs = epilogue == TJK_EPI_BIAS_RESIDUAL ? 4 : es;
  if (((uintptr_t)a & 15) || ((uintptr_t)w & 15) || ((uintptr_t)c & (4 * cs - 1)) || ((uintptr_t)bias & (4 * es - 1)))
    return fail(TJK_EUNSUPPORTED, "tjk_gemm_bias: misaligned pointer");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  switch (dtype) {
    case TJK_F32:
      return gemm_checked<float>(a, lda, w, ldw, bias, c, ldc, m, n, k, epilogue, plan_id, s);
    case TJK_F16:
      return gemm_checked<f16>(a, lda, w, ldw, bias, c, ldc, m, n, k, epilogue, plan_id, s);
    default:
      return gemm_checked<bf16>(a, lda, w, ldw, bias, c, ldc, m, n, k, epilogue, plan_id, s);
  }
}

extern "C" int tjk_gemm_bias_residual_from(const void* a, int64_t lda, const void* w, int64_t ldw,
                                           const void* bias, float* c, int64_t ldc,
                                           int64_t m, int64_t n, int64_t k,
                                           const void* x, int64_t ld_x, int64_t x_rows,
                                           const int32_t* rows, int* index_errors,
                                           int dtype, int plan_id, void* stream) {
  if (m < 0 || n < 0 || k < 0 || x_rows < 0) return fail(TJK_EINVAL, "tjk_gemm_bias_residual_from: negative shape");
  if (m == 0 || n == 0) return TJK_OK;
  // x is read only at rows below x_rows: it may be NULL when there are none
  if (!a || !w || !c || (!x && x_rows > 0)) return fail(TJK_EINVAL, "tjk_gemm_bias_residual_from: null pointer");
  if (m > INT32_MAX || n > INT32_MAX || k > INT32_MAX)
    return fail(TJK_EUNSUPPORTED, "tjk_gemm_bias_residual_from: shape exceeds int32");
  if (dtype != TJK_F32 && dtype != TJK_F16 && dtype != TJK_BF16)
    return fail(TJK_EINVAL, "tjk_gemm_bias_residual_from: bad dtype %d", dtype);
  const int es = dtype_size(dtype), vec = 16 / es;
  if (k % vec) return fail(TJK_EUNSUPPORTED, "tjk_gemm_bias_residual_from: k=%lld must be a multiple of %d", (long long)k, vec);
  if (n % 4) return fail(TJK_EUNSUPPORTED, "tjk_gemm_bias_residual_from: n=%lld must be a multiple of 4", (long long)n);
  if (lda < k || ldw < k || ldc < n || ld_x < n)
    return fail(TJK_EINVAL, "tjk_gemm_bias_residual_from: leading dimension too small");
  if (lda % vec || ldw % vec) return fail(TJK_EUNSUPPORTED, "tjk_gemm_bias_residual_from: lda/ldw must be multiples of %d", vec);
  if (ldc % 4 || ld_x % 4) return fail(TJK_EUNSUPPORTED, "tjk_gemm_bias_residual_from: ldc/ld_x must be multiples of 4");
  if (((uintptr_t)a & 15) || ((uintptr_t)w & 15) || ((uintptr_t)c & 15) || ((uintptr_t)bias & (4 * es - 1)) ||
      ((uintptr_t)x & (4 * es - 1)) || ((uintptr_t)rows & 3) || ((uintptr_t)index_errors & 3))
    return fail(TJK_EUNSUPPORTED, "tjk_gemm_bias_residual_from: misaligned pointer");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const ResSrc src{x, ld_x, rows, x_rows, index_errors};
  switch (dtype) {
    case TJK_F32:
      return gemm_checked<float>(a, lda, w, ldw, bias, c, ldc, m, n, k, kEpiResidualFrom, plan_id, s, src);
    case TJK_F16:
      return gemm_checked<f16>(a, lda, w, ldw, bias, c, ldc, m, n, k, kEpiResidualFrom, plan_id, s, src);
    default:
      return gemm_checked<bf16>(a, lda, w, ldw, bias, c, ldc, m, n, k, kEpiResidualFrom, plan_id, s, src);
  }
}
