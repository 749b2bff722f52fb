// Tile shapes of the MFMA GEMM and the launch interface between the C ABI
// (nsw_gemm.hip) and the kernel instantiations (nsw_gemm_kernel.h).
#pragma once

#include <type_traits>

#include "nsw_gemm_common.h"

namespace nsw {

// Tile of one workgroup: WGM x WGN wavefronts, each owning MB x NB blocks of
// 16 x 16 results (64 columns wide), so BM x BN results in all.  LDS_ is the
// share of the CU's 160 KB that one workgroup may take (and so how many run
// on a CU).  NST: stages of the operand ring (ring main loop).
constexpr int ROWB = 128;           // k bytes per row and LDS stage (two MFMA steps)
constexpr int STEPB = 64;           // k bytes per row consumed by one bf16 MFMA step
template <int WGM_, int WGN_, int MB_, int NST_, int LDS_>
struct TileCfg {
  static constexpr int WGM = WGM_, WGN = WGN_, MB = MB_, NB = 4, NST = NST_, LDS = LDS_;
  static constexpr int WTM = MB * 16, WTN = NB * 16;       // wave tile
  static constexpr int BM = WGM * WTM, BN = WGN * WTN;     // workgroup tile
  static constexpr int NW = WGM * WGN;                     // wavefronts per workgroup
  static constexpr int MINW = NW * (160 * 1024 / LDS) / 4; // waves per SIMD that LDS allows
  static constexpr int SLOT = (BM + BN) * ROWB;            // one stage of the ring
};
// 256 x 256, one workgroup of 8 wavefronts per CU: the large problems
using BigTile = TileCfg<2, 4, 8, 2, 160 * 1024>;

// Launches gemm_kernel<T, EPI, PRE, TC> (shapes and alignment checked by the
// caller).  Defined in nsw_gemm_kernel.h, instantiated by one source per dtype
// and tile size.
template <typename T, int EPI, int PRE, class TC>
int launch_tile(const void* x, const void* w, void* y, int64_t M, int64_t N, int64_t K, const EpiArgs& ea,
                hipStream_t st, const char* what);

// Every (epilogue, operand fusion) pair of the C ABI.
#define NSW_GEMM_FORMS(F)                                                                                            \
  F(EPI_NONE, PRE_NONE) F(EPI_BIAS, PRE_NONE) F(EPI_BIAS_GELU, PRE_NONE) F(EPI_BIAS_GELU_TANH, PRE_NONE)             \
  F(EPI_BIAS_RESIDUAL, PRE_NONE) F(EPI_WINDOW_RESIDUAL, PRE_NONE) F(EPI_SCATTER_RESIDUAL, PRE_NONE)                  \
  F(EPI_REMAP_RESIDUAL, PRE_NONE) F(EPI_RES_SUMSQ, PRE_NONE) F(EPI_TOKEN_RESIDUAL, PRE_NONE) F(EPI_UNPATCH, PRE_NONE) \
  F(EPI_QKV_HN4, PRE_NONE) F(EPI_QKV_HN8, PRE_NONE) F(EPI_QKV_HN16, PRE_NONE) F(EPI_QKV_HN32, PRE_NONE)              \
  F(EPI_QKV_HN64, PRE_NONE) F(EPI_NONE, PRE_ROWSCALE) F(EPI_BIAS, PRE_ROWSCALE) F(EPI_BIAS_GELU, PRE_ROWSCALE)       \
  F(EPI_BIAS_GELU_TANH, PRE_ROWSCALE) F(EPI_BIAS_RESIDUAL, PRE_ROWSCALE) F(EPI_QKV_HN4, PRE_ROWSCALE)                \
  F(EPI_QKV_HN8, PRE_ROWSCALE) F(EPI_QKV_HN16, PRE_ROWSCALE) F(EPI_QKV_HN32, PRE_ROWSCALE)                           \
  F(EPI_QKV_HN64, PRE_ROWSCALE)

}  // namespace nsw
