// GEMM instances: bf16, big tiles.
#include "nsw_gemm_kernel.h"

#define NSW_GEMM_T bf16
#define NSW_GEMM_SIZE Big

namespace nsw {
NSW_GEMM_FORMS(NSW_GEMM_INSTANCE)
}  // namespace nsw

using namespace nsw;

extern "C" int nsw_gemm_read_stamps(void* host, size_t bytes) {
#if NSW_GEMM_STAMPS
  NSW_CHECK_ARG(host != nullptr && bytes <= sizeof(uint64_t) * 8 * NSW_STAMP_TILES,
                "nsw_gemm_read_stamps: at most %zu bytes", sizeof(uint64_t) * 8 * (size_t)NSW_STAMP_TILES);
  if (hipMemcpyFromSymbol(host, HIP_SYMBOL(nsw_gemm_stamps), bytes, 0, hipMemcpyDeviceToHost) != hipSuccess)
    return set_error(NSW_ERR_HIP, "nsw_gemm_read_stamps: hipMemcpyFromSymbol failed");
  return 0;
#else
  (void)host; (void)bytes;
  return set_error(NSW_ERR_UNSUPPORTED, "nsw_gemm_read_stamps: library built without phase stamps (build.py --stamps)");
#endif
}

