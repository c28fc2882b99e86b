// The GEMM kernels of one element type (float).
#include "gemm_kernels.h"

namespace tjk {
template int run_gemm<float>(int, int, const GemmArgs&);
}  // namespace tjk
