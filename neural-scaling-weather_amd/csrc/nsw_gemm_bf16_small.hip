// GEMM instances: bf16, small tiles.
#undef NSW_GEMM_STAMPS
#include "nsw_gemm_kernel.h"

#define NSW_GEMM_T bf16
#define NSW_GEMM_SIZE Small

namespace nsw {
NSW_GEMM_FORMS(NSW_GEMM_INSTANCE)
}  // namespace nsw
