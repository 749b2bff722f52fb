// MFMA GEMM y[M,N] = epilogue(x[M,K] . w[N,K]^T): the C ABI and the choice of
// the tile (kernel: nsw_gemm_kernel.h).
#include <algorithm>
#include <cmath>

#include "nsw_gemm_tiles.h"

namespace nsw {

// Tile size by estimated time: rounds of workgroups over the chip's slots, a
// round of K costing fa + fb K us when every slot is taken and pa + pb K while
// at most the share f0 of the slots is (between them linear).  The constants
// are fits to measured times (M 648 - 129600, N 32 - 4096, K 32 - 2048, bias
// epilogue, within ~15%); 256 x 256 stays unless a smaller tile is estimated 7%
// faster, since its epilogues are the tuned ones.  The row epilogues go by the same
// constants: their pick was the fastest or within 10% of it at 22 sizes of both
// dtypes.  Measured, us, 256 x 256 / 128 x 128 / 64 x 128, bias epilogue:
//   bf16   648 x  128, K  512: 13.1 /  7.9 /  5.9    16200 x  192, K  768: 16.9 / 10.7 /  9.8
//   bf16  8100 x 1024, K 1024: 22.6 / 18.4 / 25.7    64800 x  512, K  512: 36.2 / 43.6 / 52.7
//   fp32   648 x  128, K  512: 45.9 / 25.5 / 19.9    16200 x  192, K  768: 71.6 / 43.4 / 40.2
//   fp32  8100 x 1024, K 1024: 97.6 / 76.3 / 97.0    32400 x  512, K  512: 58.8 / 77.5 / 91.7
struct TileCost {
  int64_t bm, bn;
  double slots, fa, fb, pa, pb, f0;
  double us(int64_t M, int64_t N, int64_t K) const {
    const double t = (double)(((M + bm - 1) / bm) * ((N + bn - 1) / bn)) / slots;
    const double r = std::floor(t), f = t - r, full = fa + fb * (double)K, part = pa + pb * (double)K;
    return r * full + (f > 0 ? part + std::max(0.0, f - f0) / (1 - f0) * (full - part) : 0);
  }
};

template <typename T, int EPI>
static TileSize pick_tile(int64_t M, int64_t N, int64_t K, const EpiArgs& ea) {
  using C = TileChoice<T, EPI>;
  constexpr bool F32 = sizeof(T) == 4;
  if (EPI == EPI_UNPATCH && ea.img_p == 16) return TILE_BIG;   // a patch of one channel is 256 columns
  constexpr TileCost big = F32 ? TileCost{256, 256, 256, 18, .0795, 9.5, .0605, 0} : TileCost{256, 256, 256, 8.5, .0234, 5.5, .015, 0};
  constexpr TileCost mid = F32 ? TileCost{C::Mid::BM, C::Mid::BN, 512, 8, .0537, 6, .0324, .4}
                               : TileCost{C::Mid::BM, C::Mid::BN, 512, 4.5, .0152, 3.6, .0088, .4};
  constexpr TileCost small = F32 ? TileCost{C::Small::BM, C::Small::BN, 768, 5, .051, 4.3, .0252, .3}
                                 : TileCost{C::Small::BM, C::Small::BN, 512, 2.3, .0099, 3.1, .0062, .4};
  const double b = big.us(M, N, K), m = mid.us(M, N, K), s = small.us(M, N, K);
  if (std::min(m, s) > 0.93 * b) return TILE_BIG;
  return s < m ? TILE_SMALL : TILE_MID;
}

template <typename T, int EPI, int PRE>
static int launch_gemm(const void* x, const void* w, void* y, int64_t M, int64_t N, int64_t K, const EpiArgs& ea,
                hipStream_t st, const char* what) {
  constexpr int KT = STEPB / sizeof(T);   // k granule: 32 (bf16) / 16 (f32)
  NSW_CHECK_ARG(M > 0 && N > 0 && K > 0, "%s: M, N, K must be positive", what);
  NSW_CHECK_ARG(K % KT == 0, "%s: K=%lld must be a multiple of %d", what, (long long)K, KT);
  NSW_CHECK_ARG(N % 8 == 0, "%s: N=%lld must be a multiple of 8", what, (long long)N);
  NSW_CHECK_ARG(M < (1LL << 31) && N < (1LL << 31) && K < (1LL << 31), "%s: dims too large", what);
  NSW_CHECK_ARG((uint64_t)M * K * sizeof(T) < (1ULL << 31) && (uint64_t)N * K * sizeof(T) < (1ULL << 31),
                "%s: operands above 2 GiB are not supported (32-bit buffer offsets)", what);
  NSW_CHECK_ARG(((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0 && ((uintptr_t)y % 16) == 0 &&
                    ((uintptr_t)ea.residual % 16) == 0,
                "%s: x, w, y and residual must be 16-byte aligned", what);
  EpiArgs eg = ea;
  if constexpr (EPI == EPI_BIAS_GELU || EPI == EPI_BIAS_GELU_TANH) {
    // the MLP's first GEMM: tile groups of ~128 tiles (8 row blocks x 16
    // column blocks at config 2, 16 x 8 at config 4: each measured 5% faster
    // than the other height on its shape)
    if (eg.group_m == 0) eg.group_m = (int)std::max<int64_t>(8, std::min<int64_t>(32, 128 / ((N + 255) / 256)));
  }
  using C = TileChoice<T, EPI>;
  switch (pick_tile<T, EPI>(M, N, K, ea)) {
    case TILE_BIG: return launch_tile<T, EPI, PRE, BigTile>(x, w, y, M, N, K, eg, st, what);
    case TILE_MID: return launch_tile<T, EPI, PRE, typename C::Mid>(x, w, y, M, N, K, eg, st, what);
    default: return launch_tile<T, EPI, PRE, typename C::Small>(x, w, y, M, N, K, eg, st, what);
  }
}

template <int EPI, int PRE = PRE_NONE>
static int dispatch_gemm(int dtype, const void* x, const void* w, void* y, int64_t M, int64_t N,
                         int64_t K, const EpiArgs& ea, void* stream, const char* what) {
  hipStream_t st = (hipStream_t)stream;
  if (dtype == NSW_DTYPE_BF16) return launch_gemm<bf16, EPI, PRE>(x, w, y, M, N, K, ea, st, what);
  if (dtype == NSW_DTYPE_F32) return launch_gemm<float, EPI, PRE>(x, w, y, M, N, K, ea, st, what);
  return set_error(NSW_ERR_INVALID, "%s: unknown dtype %d", what, dtype);
}


int check_geom(int64_t B, int64_t T, int64_t H, int64_t W, int64_t ws0, int64_t ws1, const char* what);

int gemm_qkv(const void* x, const void* wqkv, const void* bqkv, const void* qn_w, const void* kn_w,
             float eps, void* qkv, int64_t M, int64_t C, int64_t num_heads, int dtype, void* stream) {
  const char* what = "nsw_qkv_projection";
  NSW_CHECK_ARG(num_heads > 0 && C % num_heads == 0, "%s: C=%lld not divisible by num_heads=%lld", what,
                (long long)C, (long long)num_heads);
  const int64_t hd = C / num_heads;
  NSW_CHECK_ARG(C % 16 == 0, "%s: C=%lld must be a multiple of 16", what, (long long)C);
  NSW_CHECK_ARG(hd == 4 || hd == 8 || hd == 16 || hd == 32 || hd == 64,
                "%s: head_dim=%lld unsupported (4, 8, 16, 32, 64)", what, (long long)hd);
  NSW_CHECK_ARG(bqkv && qn_w && kn_w, "%s: bias and norm weights are required", what);
  EpiArgs ea{};
  ea.bias = bqkv; ea.qn_w = qn_w; ea.kn_w = kn_w; ea.eps = eps; ea.C = (int)C;
  ea.group_m = 4;
  if (hd == 64) return dispatch_gemm<EPI_QKV_HN64>(dtype, x, wqkv, qkv, M, 3 * C, C, ea, stream, what);
  if (hd == 32) return dispatch_gemm<EPI_QKV_HN32>(dtype, x, wqkv, qkv, M, 3 * C, C, ea, stream, what);
  if (hd == 8) return dispatch_gemm<EPI_QKV_HN8>(dtype, x, wqkv, qkv, M, 3 * C, C, ea, stream, what);
  if (hd == 4) return dispatch_gemm<EPI_QKV_HN4>(dtype, x, wqkv, qkv, M, 3 * C, C, ea, stream, what);
  return dispatch_gemm<EPI_QKV_HN16>(dtype, x, wqkv, qkv, M, 3 * C, C, ea, stream, what);
}

// Partial sums of squares per output row: one float per 512 bytes of row
// (32 lanes of 16-byte stores in the scatter epilogue).
int64_t sumsq_parts(int64_t C, int dtype) {
  const int64_t es = dtype == NSW_DTYPE_F32 ? 4 : 2;
  return (C * es + 511) / 512;
}

int gemm_proj_scatter(const void* o, const void* wproj, const void* bproj, const void* skip, void* y,
                      int64_t B, int64_t T, int64_t H, int64_t W, int64_t C, int64_t ws0, int64_t ws1,
                      int64_t s0, int64_t s1, int dtype, void* stream, float* row_sumsq) {
  const char* what = row_sumsq ? "nsw_proj_reverse_residual_sumsq" : "nsw_proj_reverse_residual";
  int rc = check_geom(B, T, H, W, ws0, ws1, what);
  if (rc) return rc;
  NSW_CHECK_ARG(bproj && skip, "%s: bias and skip are required", what);
  NSW_CHECK_ARG(skip != (const void*)y, "%s: skip and y must not alias (rows are permuted)", what);
  EpiArgs ea{};
  ea.bias = bproj; ea.residual = skip;
  ea.geom = WinGeom::make((int)B, (int)T, (int)H, (int)W, (int)ws0, (int)ws1, (int)(s0 % H), (int)(s1 % W));
  ea.row_sumsq = row_sumsq;
  ea.nparts = (int)sumsq_parts(C, dtype);
  ea.group_m = 16;   // proj's 4 column blocks: 16-row-block groups measured 2.5% faster than 8
  return dispatch_gemm<EPI_SCATTER_RESIDUAL>(dtype, o, wproj, y, B * T * H * W, C, C, ea, stream, what);
}

// y = epi(rs . (x . w_n^T)), rs[m] = 1/sqrt(sum_p row_sumsq[m, p] / K + eps):
// RMSNorm(x) folded into the GEMM with the row statistics from x's producer.
int gemm_linear_rowscale(const void* x, const void* w_n, const void* bias, const void* residual, void* y,
                         const float* row_sumsq, int64_t nparts, int64_t M, int64_t N, int64_t K, int epilogue,
                         float eps, int dtype, void* stream) {
  const char* what = "nsw_linear_rowscale";
  NSW_CHECK_ARG(row_sumsq != nullptr && nparts > 0 && nparts <= 4096, "%s: row_sumsq [M, nparts] is required",
                what);
  NSW_CHECK_ARG(((uintptr_t)row_sumsq % 16) == 0, "%s: row_sumsq must be 16-byte aligned", what);
  EpiArgs ea{};
  ea.bias = bias; ea.residual = residual; ea.eps = eps;
  ea.row_sumsq = const_cast<float*>(row_sumsq);
  ea.nparts = (int)nparts;
  if (epilogue != NSW_EPI_NONE) NSW_CHECK_ARG(bias != nullptr, "%s: epilogue %d needs a bias", what, epilogue);
  switch (epilogue) {
    case NSW_EPI_NONE: return dispatch_gemm<EPI_NONE, PRE_ROWSCALE>(dtype, x, w_n, y, M, N, K, ea, stream, what);
    case NSW_EPI_BIAS: return dispatch_gemm<EPI_BIAS, PRE_ROWSCALE>(dtype, x, w_n, y, M, N, K, ea, stream, what);
    case NSW_EPI_BIAS_GELU:
      return dispatch_gemm<EPI_BIAS_GELU, PRE_ROWSCALE>(dtype, x, w_n, y, M, N, K, ea, stream, what);
    case NSW_EPI_BIAS_GELU_TANH:
      return dispatch_gemm<EPI_BIAS_GELU_TANH, PRE_ROWSCALE>(dtype, x, w_n, y, M, N, K, ea, stream, what);
    case NSW_EPI_BIAS_RESIDUAL:
      NSW_CHECK_ARG(residual != nullptr, "%s: residual epilogue needs a residual", what);
      return dispatch_gemm<EPI_BIAS_RESIDUAL, PRE_ROWSCALE>(dtype, x, w_n, y, M, N, K, ea, stream, what);
    default: return set_error(NSW_ERR_INVALID, "%s: unknown epilogue %d", what, epilogue);
  }
}

// QKV projection of rows whose RMSNorm (norm1) comes as a row scale from the
// producer's partial sums of squares: qkv[m] = headnorm(rs1[m] * (x[m] .
// wqkv_n^T) + b), wqkv_n = wqkv * norm1_w per input column, rs1 =
// 1/sqrt(sum_p row_sumsq[m, p] / C + eps).  Rows in any order.
int gemm_qkv_rowscale(const void* x, const void* wqkv_n, const void* bqkv, const void* qn_w, const void* kn_w,
                      float eps, void* qkv, const float* row_sumsq, int64_t nparts, int64_t M, int64_t C,
                      int64_t num_heads, int dtype, void* stream) {
  const char* what = "nsw_qkv_projection_rowscale";
  NSW_CHECK_ARG(num_heads > 0 && C % num_heads == 0, "%s: C=%lld not divisible by num_heads=%lld", what,
                (long long)C, (long long)num_heads);
  const int64_t hd = C / num_heads;
  NSW_CHECK_ARG(C % 16 == 0, "%s: C=%lld must be a multiple of 16", what, (long long)C);
  NSW_CHECK_ARG(hd == 4 || hd == 8 || hd == 16 || hd == 32 || hd == 64,
                "%s: head_dim=%lld unsupported (4, 8, 16, 32, 64)", what, (long long)hd);
  NSW_CHECK_ARG(bqkv && qn_w && kn_w, "%s: bias and norm weights are required", what);
  NSW_CHECK_ARG(row_sumsq != nullptr && nparts > 0 && nparts <= 4096 && ((uintptr_t)row_sumsq % 16) == 0,
                "%s: row_sumsq [M, nparts] (16-byte aligned) is required", what);
  EpiArgs ea{};
  ea.bias = bqkv; ea.qn_w = qn_w; ea.kn_w = kn_w; ea.eps = eps; ea.C = (int)C;
  ea.group_m = 4;
  ea.row_sumsq = const_cast<float*>(row_sumsq);
  ea.nparts = (int)nparts;
  if (hd == 64) return dispatch_gemm<EPI_QKV_HN64, PRE_ROWSCALE>(dtype, x, wqkv_n, qkv, M, 3 * C, C, ea, stream, what);
  if (hd == 32) return dispatch_gemm<EPI_QKV_HN32, PRE_ROWSCALE>(dtype, x, wqkv_n, qkv, M, 3 * C, C, ea, stream, what);
  if (hd == 8) return dispatch_gemm<EPI_QKV_HN8, PRE_ROWSCALE>(dtype, x, wqkv_n, qkv, M, 3 * C, C, ea, stream, what);
  if (hd == 4) return dispatch_gemm<EPI_QKV_HN4, PRE_ROWSCALE>(dtype, x, wqkv_n, qkv, M, 3 * C, C, ea, stream, what);
  return dispatch_gemm<EPI_QKV_HN16, PRE_ROWSCALE>(dtype, x, wqkv_n, qkv, M, 3 * C, C, ea, stream, what);
}

// y[remap(m)] = x[m] . w^T + bias + residual[m], the stored rows' partial
// sums of squares (one float per 512 bytes of row) into row_sumsq at the
// same rows where asked.  map_mode 0: remap(m) = m (row_sumsq required); 1:
// the token of window-order row m of the image geometry (B, T, H, W, ws,
// shift s) (no row sums); 2: that token's row in the window order of the
// same image rolled by (sa, sb), the next block's (row_sumsq required).
int gemm_linear_remap(const void* x, const void* w, const void* bias, const void* residual, void* y,
                      float* row_sumsq, int64_t M, int64_t N, int64_t K, int map_mode, int64_t B, int64_t T,
                      int64_t H, int64_t W, int64_t ws0, int64_t ws1, int64_t s0, int64_t s1, int64_t sa,
                      int64_t sb, int dtype, void* stream) {
  const char* what = "nsw_linear_remap_residual";
  NSW_CHECK_ARG(bias && residual, "%s: bias and residual are required", what);
  NSW_CHECK_ARG(residual != (const void*)y, "%s: residual and y must not alias", what);
  NSW_CHECK_ARG(map_mode >= 0 && map_mode <= 3, "%s: map_mode must be 0, 1, 2 or 3", what);
  NSW_CHECK_ARG((row_sumsq != nullptr) == (map_mode != 1),
                "%s: row sums of squares are written for map modes 0, 2 and 3, and required there", what);
  EpiArgs ea{};
  ea.bias = bias; ea.residual = residual;
  if (map_mode != 0) {
    int rc = check_geom(B, T, H, W, ws0, ws1, what);
    if (rc) return rc;
    NSW_CHECK_ARG(M == B * T * H * W, "%s: M must be B*T*H*W for a row map", what);
    ea.geom = WinGeom::make((int)B, (int)T, (int)H, (int)W, (int)ws0, (int)ws1, (int)(s0 % H), (int)(s1 % W));
    const int64_t a = ((sa % H) + H) % H, b = ((sb % W) + W) % W;
    ea.dh = (int)(((ea.geom.s0 - a) % H + H) % H);
    ea.dw = (int)(((ea.geom.s1 - b) % W + W) % W);
  }
  ea.row_sumsq = row_sumsq;
  ea.nparts = (int)sumsq_parts(N, dtype);
  if (row_sumsq) NSW_CHECK_ARG(((uintptr_t)row_sumsq % 4) == 0, "%s: row_sumsq must be 4-byte aligned", what);
  if (map_mode == 0) {
    ea.group_m = N <= 1024 ? 16 : 0;   // proj-shaped (few column blocks): 16-row-block groups
    return dispatch_gemm<EPI_RES_SUMSQ>(dtype, x, w, y, M, N, K, ea, stream, what);
  }
  if (map_mode == 1) return dispatch_gemm<EPI_TOKEN_RESIDUAL>(dtype, x, w, y, M, N, K, ea, stream, what);
  if (map_mode == 3) return dispatch_gemm<EPI_WINDOW_RESIDUAL>(dtype, x, w, y, M, N, K, ea, stream, what);
  return dispatch_gemm<EPI_REMAP_RESIDUAL>(dtype, x, w, y, M, N, K, ea, stream, what);
}

}  // namespace nsw

using namespace nsw;

extern "C" int nsw_linear(const void* x, const void* w, const void* bias, const void* residual, void* y,
                          int64_t M, int64_t N, int64_t K, int epilogue, int dtype, void* stream) {
  const char* what = "nsw_linear";
  EpiArgs ea{};
  ea.bias = bias; ea.residual = residual;
  if (epilogue != NSW_EPI_NONE) NSW_CHECK_ARG(bias != nullptr, "%s: epilogue %d needs a bias", what, epilogue);
  switch (epilogue) {
    case NSW_EPI_NONE: return dispatch_gemm<EPI_NONE>(dtype, x, w, y, M, N, K, ea, stream, what);
    case NSW_EPI_BIAS: return dispatch_gemm<EPI_BIAS>(dtype, x, w, y, M, N, K, ea, stream, what);
    case NSW_EPI_BIAS_GELU: return dispatch_gemm<EPI_BIAS_GELU>(dtype, x, w, y, M, N, K, ea, stream, what);
    case NSW_EPI_BIAS_GELU_TANH:
      return dispatch_gemm<EPI_BIAS_GELU_TANH>(dtype, x, w, y, M, N, K, ea, stream, what);
    case NSW_EPI_BIAS_RESIDUAL:
      NSW_CHECK_ARG(residual != nullptr, "%s: residual epilogue needs a residual", what);
      return dispatch_gemm<EPI_BIAS_RESIDUAL>(dtype, x, w, y, M, N, K, ea, stream, what);
    default: return set_error(NSW_ERR_INVALID, "%s: unknown epilogue %d", what, epilogue);
  }
}

extern "C" int nsw_qkv_projection(const void* x, const void* wqkv, const void* bqkv, const void* qn_w,
                                  const void* kn_w, float eps, void* qkv, int64_t M, int64_t C,
                                  int64_t num_heads, int dtype, void* stream) {
  return gemm_qkv(x, wqkv, bqkv, qn_w, kn_w, eps, qkv, M, C, num_heads, dtype, stream);
}

extern "C" int nsw_proj_reverse_residual(const void* o, const void* wproj, const void* bproj,
                                         const void* skip, void* y, int64_t B, int64_t T, int64_t H,
                                         int64_t W, int64_t C, int64_t ws0, int64_t ws1, int64_t s0,
                                         int64_t s1, int dtype, void* stream) {
  return gemm_proj_scatter(o, wproj, bproj, skip, y, B, T, H, W, C, ws0, ws1, s0, s1, dtype, stream, nullptr);
}

extern "C" int nsw_gemm_tile_rows(int64_t M, int64_t N, int64_t K, int row_epilogue, int dtype) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  auto rows = [](TileSize t, int big, int mid, int small) { return t == TILE_BIG ? big : t == TILE_MID ? mid : small; };
  const EpiArgs ea{};
  if (dtype == NSW_DTYPE_F32)
    return rows(pick_tile<float, EPI_NONE>(M, N, K, ea), BigTile::BM, MidTile::BM, SmallF32Tile::BM);
  if (dtype != NSW_DTYPE_BF16) return 0;
  if (row_epilogue) return rows(pick_tile<bf16, EPI_RES_SUMSQ>(M, N, K, ea), BigTile::BM, MidRowTile::BM, SmallRowTile::BM);
  return rows(pick_tile<bf16, EPI_NONE>(M, N, K, ea), BigTile::BM, MidTile::BM, SmallTile::BM);
}

extern "C" int64_t nsw_row_sumsq_parts(int64_t C, int dtype) { return C > 0 ? sumsq_parts(C, dtype) : 0; }

extern "C" int nsw_proj_reverse_residual_sumsq(const void* o, const void* wproj, const void* bproj,
                                               const void* skip, void* y, float* row_sumsq, int64_t B,
                                               int64_t T, int64_t H, int64_t W, int64_t C, int64_t ws0,
                                               int64_t ws1, int64_t s0, int64_t s1, int dtype, void* stream) {
  NSW_CHECK_ARG(row_sumsq != nullptr, "nsw_proj_reverse_residual_sumsq: row_sumsq is required");
  return gemm_proj_scatter(o, wproj, bproj, skip, y, B, T, H, W, C, ws0, ws1, s0, s1, dtype, stream, row_sumsq);
}

extern "C" int nsw_linear_rowscale(const void* x, const void* w_n, const void* bias, const void* residual,
                                   void* y, const float* row_sumsq, int64_t nparts, int64_t M, int64_t N,
                                   int64_t K, int epilogue, float eps, int dtype, void* stream) {
  return gemm_linear_rowscale(x, w_n, bias, residual, y, row_sumsq, nparts, M, N, K, epilogue, eps, dtype, stream);
}

extern "C" int nsw_qkv_projection_rowscale(const void* x, const void* wqkv_n, const void* bqkv, const void* qn_w,
                                           const void* kn_w, float eps, void* qkv, const float* row_sumsq,
                                           int64_t nparts, int64_t M, int64_t C, int64_t num_heads, int dtype,
                                           void* stream) {
  return gemm_qkv_rowscale(x, wqkv_n, bqkv, qn_w, kn_w, eps, qkv, row_sumsq, nparts, M, C, num_heads, dtype,
                           stream);
}

// The forecast head with its layout fused in: image = unpatchify(x . w_perm^T)
// (models/swin.py:286-299), w_perm the head weight with its rows permuted
// from the reference's (dy p + dx) C_out + c to c p^2 + dy p + dx.
int gemm_head_unpatchify(const void* x, const void* w_perm, void* out, int64_t B, int64_t C_out, int64_t H,
                         int64_t W, int64_t p, int64_t K, int64_t out_bstride, int dtype, int out_dtype,
                         void* stream) {
  const char* what = "nsw_head_unpatchify";
  NSW_CHECK_ARG(B > 0 && C_out > 0 && H > 0 && W > 0 && K > 0, "%s: B, C_out, H, W, K must be positive", what);
  NSW_CHECK_ARG(p == 1 || p == 2 || p == 4 || p == 8 || p == 16, "%s: p=%lld must be 1, 2, 4, 8 or 16", what,
                (long long)p);
  NSW_CHECK_ARG(H % p == 0 && W % p == 0, "%s: H=%lld, W=%lld not divisible by p=%lld", what, (long long)H,
                (long long)W, (long long)p);
  NSW_CHECK_ARG(dtype == NSW_DTYPE_BF16 || dtype == NSW_DTYPE_F32, "%s: unknown dtype %d", what, dtype);
  NSW_CHECK_ARG(out_dtype == dtype || out_dtype == NSW_DTYPE_F32,
                "%s: the image is in the GEMM's dtype or float32 (got %d for %d)", what, out_dtype, dtype);
  NSW_CHECK_ARG(out_bstride >= C_out * H * W && out_bstride % p == 0,
                "%s: out_bstride must cover one frame and be a multiple of p", what);
  const int64_t oes = out_dtype == NSW_DTYPE_F32 ? 4 : 2;
  NSW_CHECK_ARG(((uintptr_t)out % (uintptr_t)std::min<int64_t>(16, p * oes)) == 0,
                "%s: out must be aligned to min(16, p * element size) bytes", what);
  NSW_CHECK_ARG(B * out_bstride < (1LL << 40) && H * W < (1LL << 31), "%s: image too large", what);
  EpiArgs ea{};
  ea.img = out;
  ea.img_bstride = out_bstride;
  ea.img_C = (int)C_out; ea.img_H = (int)H; ea.img_W = (int)W; ea.img_p = (int)p;
  ea.img_f32 = out_dtype == NSW_DTYPE_F32 && dtype == NSW_DTYPE_BF16;
  const int64_t M = B * (H / p) * (W / p);
  return dispatch_gemm<EPI_UNPATCH>(dtype, x, w_perm, nullptr, M, C_out * p * p, K, ea, stream, what);
}

extern "C" int nsw_head_unpatchify(const void* x, const void* w_perm, void* out, int64_t B, int64_t C_out,
                                   int64_t H, int64_t W, int64_t p, int64_t K, int64_t out_bstride, int dtype,
                                   int out_dtype, void* stream) {
  return gemm_head_unpatchify(x, w_perm, out, B, C_out, H, W, p, K, out_bstride, dtype, out_dtype, stream);
}

extern "C" int nsw_linear_remap_residual(const void* x, const void* w, const void* bias, const void* residual,
                                         void* y, float* row_sumsq, int64_t M, int64_t N, int64_t K, int map_mode,
                                         int64_t B, int64_t T, int64_t H, int64_t W, int64_t ws0, int64_t ws1,
                                         int64_t s0, int64_t s1, int64_t sa, int64_t sb, int dtype,
                                         void* stream) {
  return gemm_linear_remap(x, w, bias, residual, y, row_sumsq, M, N, K, map_mode, B, T, H, W, ws0, ws1, s0, s1,
                           sa, sb, dtype, stream);
}
