// The GEMM kernels of one element type (bf16).
#include "gemm_kernels.h"

namespace tjk {
template int run_gemm<bf16>(int, int, const GemmArgs&);
}  // namespace tjk
