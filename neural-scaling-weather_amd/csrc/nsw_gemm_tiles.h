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
// Smaller tiles of 4 wavefronts, two or three workgroups per CU, for problems
// that leave CUs idle at 256 x 256 (pick_tile).  The Row tiles are 256 columns
// wide (512 bytes of bf16 row, the unit of the row sums of squares).  Deeper
// rings with one workgroup per CU were slower at every size: with few
// wavefronts a stage's time is its chain of barrier, LDS reads and issue, not
// the copies' latency; 8 wavefronts of half the rows per 128 x 128 tile
// measured the same.
using MidTile = TileCfg<2, 2, 4, 2, 80 * 1024>;         // 128 x 128
using MidRowTile = TileCfg<1, 4, 4, 2, 80 * 1024>;      // 64 x 256
using SmallTile = TileCfg<2, 2, 2, 3, 80 * 1024>;       // 64 x 128, bf16
using SmallRowTile = TileCfg<1, 4, 2, 2, 80 * 1024>;    // 32 x 256, bf16
using SmallF32Tile = TileCfg<2, 2, 2, 2, 53 * 1024>;    // 64 x 128, fp32

// Epilogues that store rows through a map or write row sums of squares: in
// bf16 these take the Row tiles (a 512-byte part of a row lies in one tile).
constexpr bool row_epi(int epi) {
  return epi == EPI_SCATTER_RESIDUAL || epi == EPI_REMAP_RESIDUAL || epi == EPI_WINDOW_RESIDUAL ||
         epi == EPI_RES_SUMSQ || epi == EPI_TOKEN_RESIDUAL;
}

enum TileSize { TILE_BIG, TILE_MID, TILE_SMALL };
template <typename T, int EPI> struct TileChoice {
  static constexpr bool ROW = sizeof(T) == 2 && row_epi(EPI);
  using Big = BigTile;
  using Mid = std::conditional_t<ROW, MidRowTile, MidTile>;
  using Small = std::conditional_t<sizeof(T) == 4, SmallF32Tile, std::conditional_t<ROW, SmallRowTile, SmallTile>>;
};

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
