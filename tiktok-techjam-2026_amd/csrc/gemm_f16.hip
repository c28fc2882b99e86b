// The GEMM kernels of one element type (f16).
#include "gemm_kernels.h"

namespace tjk {
template int run_gemm<f16>(int, int, const GemmArgs&);
}  // namespace tjk
