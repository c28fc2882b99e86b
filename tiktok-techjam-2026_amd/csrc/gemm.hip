// Entry points of the GEMM (tjk_gemm_bias, tjk_gemm_bias_residual_from):
// argument checks and the default tile choice.  The kernels are in
// gemm_kernels.h, compiled once per element type.

#include "gemm_plans.h"

namespace tjk {

static bool dtl_ok(const GemmPlan& p, int64_t k, int64_t lda, int64_t ldw, int es) {
  return k % (p.bkb / es) == 0 && (lda * es) % 16 == 0 && (ldw * es) % 16 == 0;
}

// Default tile choice.  For shapes the direct-to-LDS kernel takes, the
// measured rule above; otherwise (odd K, misaligned rows) the staged plan
// minimising (full-chip rounds of 256 workgroups) x (tile area / prior).
template <typename T>
static int auto_plan(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldw) {
  int count;
  const GemmPlan* p = plans<T>(&count);
  if (sizeof(T) == 2 && dtl_ok(p[7], K, lda, ldw, sizeof(T))) {
    // 256 x 256 tiles run one per CU: worth it when they come within 10% of
    // whole rounds of the 256 CUs.  Measured (bf16): 8192 x 2048 x 8192 (one
    // round) 193 us as plan 33, 216 as 8, 253 as 7; 8192 x 8192 x 2048 231 /
    // 244 / 274; 5430 x 3072 x 1024 (264 tiles) 55 / 54 / 47.
    const int64_t t256 = ((M + 255) / 256) * ((N + 255) / 256);
    const int64_t t128 = ((M + 127) / 128) * ((N + 127) / 128);
    if (10 * t256 >= 9 * 256 * ((t256 + 255) / 256)) return 33;
    if (t128 >= 128) return 7;
    return 9;
  }
  int best = 0;
  double best_cost = 1e300;
  for (int i = 0; i < count; ++i) {
    if (p[i].kind != kStaged && !dtl_ok(p[i], K, lda, ldw, sizeof(T))) continue;
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
  if (plan == -1) plan = auto_plan<T>(m, n, k, lda, ldw);
  if (p[plan].kind != kStaged && !dtl_ok(p[plan], k, lda, ldw, sizeof(T)))
    return fail(TJK_EUNSUPPORTED, "tjk_gemm_bias: plan %d needs k %% %d == 0", plan, (int)(p[plan].bkb / sizeof(T)));
  if (p[plan].kind != kStaged && ((int64_t)p[plan].bm * lda * (int64_t)sizeof(T) > INT32_MAX ||
                                  (int64_t)p[plan].bn * ldw * (int64_t)sizeof(T) > INT32_MAX))
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
