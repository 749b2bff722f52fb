// Kernel of the MFMA GEMM y[M,N] = epilogue(x[M,K] . w[N,K]^T) for gfx950, with
// the Swin block's epilogues fused in: main loops, epilogues and the launch.
// Included by one source per dtype and tile size.
//
// Three tile sizes (nsw_gemm_tiles.h); this is the bf16 256 x 256 one, whose main
// loop is mainloop_256 (the smaller ones: mainloop_ring; fp32: mainloop_split2 and
// mainloop_split3).
//
// Workgroup tile 256 (m) x 256 (n), one workgroup of 8 wavefronts per CU
// (two per SIMD, so that one wave's MFMAs cover the other's LDS reads and
// waits) in a 2 (m) x 4 (n) grid, each owning a 128 x 64 sub-tile of 16x16
// fp32 accumulator blocks (128 accumulator registers per lane).  A stage holds
// 128 bytes of k (64 bf16) of the 256 x-rows and the 256 w-rows and is
// consumed as two MFMA steps of 32 bf16; x lives (bf16) in a ring of 3 slots and w in
// a ring of 2 slots of 32 KB (all 160 KB of LDS), filled at a steady 4 copies
// per wave and MFMA step (schedule at mainloop_256).  Whole 128-byte lines
// per copy.
//
// Operand staging: global -> LDS copies use gfx950's buffer_load_dwordx4 ...
// lds (direct to LDS, no VGPR staging): each instruction writes 1 KB = 8 stage
// rows of one wave's share.  Rows are XOR-swizzled in 16-byte chunks so that a
// fragment read (16 rows, same chunk) is bank-conflict free whether
// ds_read_b128 is served in 8-lane phases over 32 banks or 16-lane phases over
// 64 banks: slot = chunk ^ g(row & 15), g(r) = ((r >> 1) & 7) ^ ((r & 1) << 2).
// The MFMAs of step k run from registers while the fragments of step k+1 are
// read between them: the MFMAs go n block by n block, and the next step's
// weight fragment of an n block is read into the registers that block's
// MFMAs have just released, so the x fragments are double-buffered and the
// w fragments take one set (the register file of two waves per SIMD has no
// room for two of both).  Barriers are s_barrier behind a wait for the
// wave's own LDS accesses: __syncthreads() would add a fence that waits for
// every outstanding copy.
//
// The MFMA is issued "transposed": the A operand is the weight fragment
// (rows n) and the B operand the activation fragment (rows m), so lane l of a
// 16x16 result block holds y[m = l%16][n = 4*(l/16) + r], r = 0..3: four
// consecutive output columns, and a row's head-norm reduction needs only two
// cross-lane permutes.
//
//   bf16: v_mfma_f32_16x16x32_bf16, one instruction per 16-byte fragment pair
//   f32 : the 16-bit instructions of the same shape on operands split into two
//         or three parts (mainloop_split2, mainloop_split3)
//
// Workgroups are remapped so that each XCD (8 on MI355X, dispatched
// round-robin) works on a contiguous range of tiles, in groups of GROUP_M
// row blocks x all column blocks (column-major inside a group), so that the
// tiles in flight on an XCD share both row panels and weight panels in its L2.
#pragma once

#include "nsw_gemm_tiles.h"

// Per-tile phase stamps, compiled in only with -DNSW_GEMM_STAMPS=1 (build.py
// --stamps, which writes nsw/libnsw_stamps.so; the default library has
// none): thread 0 of each workgroup reads s_memtime when its tile starts,
// when the prologue's first stages have landed, after the main loop, after
// the first epilogue phase is staged and at the end, and stores them with
// HW_ID, XCC_ID and the workgroup id as 8 words at tile * 8 of
// nsw_gemm_stamps (the first NSW_STAMP_TILES tiles of each launch; every
// launch overwrites them).  nsw_gemm_read_stamps copies them to the host.
#ifndef NSW_GEMM_STAMPS
#define NSW_GEMM_STAMPS 0
#endif
#if NSW_GEMM_STAMPS
constexpr int NSW_STAMP_TILES = 65536;
__device__ uint64_t nsw_gemm_stamps[NSW_STAMP_TILES * 8];
#define NSW_STAMP(var) (var) = __builtin_amdgcn_s_memtime()
#else
#define NSW_STAMP(var) ((void)0)
#endif

namespace nsw {

typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
// fp32 operands run on the 16-bit matrix instructions, split into two scaled
// fp16 parts (three products) from this K on and into three bf16 parts (six
// products) below it; values that two fp16 parts do not hold are looked for one by
// one (mainloop_split2).  v_mfma_f32_16x16x4_f32 has 1/16 of their rate; on normal
// rows both forms are also closer to the 64-bit result than it was, because a sum
// takes K / 32 x 3 or x 6 roundings instead of K.  Relative error (2-norm) of x .
// w^T, x N(0, 1), w N(0, 0.02): fp32 instruction / three parts / two parts
//   K =   32: 1.0e-7 / 3.8e-8 / 8.8e-8       K =  192: 2.5e-7 / 2.0e-7 / 1.6e-7
//   K =   96: 1.8e-7 / 1.3e-7 / 1.2e-7       K = 1024: 5.7e-7 / 4.8e-7 / 3.6e-7
//   K =  128: 2.0e-7 / 1.6e-7 / 1.4e-7       K = 4096: 1.2e-6 / 1.0e-6 / 7.1e-7
// Below K = 128 three parts are as close or closer and mostly faster (us, three /
// two: 129600 x 128, K 32 17.6 / 25.8; 16200 x 192, K 96 11.8 / 13.7; 64800 x 384, K
// 112 46.8 / 59.5; 64800 x 1024, K 96 101.9 / 96.3).
// Time (us, 64800 rows, no bias), N 3072, K 1024 / N 1024, K 4096:
//   fp32 instruction                                        2829 / 3674
//   two parts, values not looked at                         1111 / 1430
//   normal rows                                             1256 / 1659
//   a column 1e4 times the others                           1605 / 2119
//   half the values zero                                    1629 / 1996
//   values of any size (three parts from the first stage)   1882 / 2394
//   GELU(2 x - 2)                                           2212 / 2491
//   a row that is not finite                                1322 / 1870
constexpr int SPLIT2_MIN_K = 128;

// bf16 256 x 256 tiles run mainloop_256.
template <typename T, class TC>
constexpr bool is_main256 = sizeof(T) == 2 && TC::BM == 256 && TC::BN == 256;

// epilogue staging of the output tile in LDS, in the output dtype: the whole
// tile when it fits beside the epilogue's parameters, else two halves; rows
// padded by 16 B so that the fragment-layout writes spread over the banks.
// The parameters (floats) follow the staging rows: bias [0, BN), q/k norm
// weights [PRM_NW, +128), row scales [PRM_RS, +BM).
template <typename T, class TC> struct Stg {
  static constexpr int PRM_NW = TC::BN, PRM_RS = TC::BN + 128;
  static constexpr int PRMB = (TC::BN + 128 + TC::BM) * 4;
  static constexpr int STRIDE = TC::BN * (int)sizeof(T) + 16;
  static constexpr int ROWS = TC::BM * STRIDE + PRMB <= TC::LDS ? TC::BM : TC::BM / 2;
  static constexpr int PASSES = TC::BM / ROWS;
  static constexpr int BYTES = ROWS * STRIDE;
  // operand ring: x in 3 and w in 2 slots (mainloop_256), else NST stages
  static constexpr int RING = is_main256<T, TC> ? 5 * 256 * ROWB : TC::NST * TC::SLOT;
  static constexpr int PARAM_LDS = BYTES;
  static constexpr int SMEM = RING > BYTES + PRMB ? RING : BYTES + PRMB;
  static_assert(SMEM <= TC::LDS, "LDS use exceeds the workgroup's share");
};

__device__ __forceinline__ void mfma_bf16(f32x4& acc, const bf16x8& a, const bf16x8& b) {
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
}

__device__ __forceinline__ void mfma_f16(f32x4& acc, const f16x8& a, const f16x8& b) {
  acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, acc, 0, 0, 0);
}

// Fragment read: 16 bytes of k chunk `chunk` of a stage row.
__device__ __forceinline__ u32x4 lds_frag(const char* stage, int row, int chunk) {
  const int slot = chunk ^ row_swizzle(row);
  return *reinterpret_cast<const u32x4*>(stage + row * ROWB + slot * 16);
}

// Main loop of the 256 x 256 tile.  Stage st holds 128 bytes of k of the 256
// x rows and the 256 w rows.  x lives in a ring of 3 slots and w in a ring of
// 2 slots of 32 KB (160 KB in all).  The copies are issued by the four waves
// of the first row half (waves 0-3, one per SIMD: NC = 8 copies of each
// operand per stage each, 64 rows); the other four waves run only LDS reads
// and MFMAs, so that on every SIMD one wave's MFMA stream is free of copy
// issue (bit-identical; 2-5% faster on the block's four GEMM shapes than
// 4 + 4 copies per wave, measured on one box; the copies on waves 4-7
// instead were 2-5% slower than 4 + 4).  A copying wave issues its copies of
// a step in the step's first two n blocks (4 each):
//   step 2s+1 (the second step of stage s, after the barrier that frees the
//              slots of stage s): w of stage s+2 into w slot s%2;
//   step 2s+2 (the first step of stage s+1): x of stage s+3 into x slot s%3,
// and the x copies (the operand with fewer sharers in L2) get 2-3 steps of
// lead, the w copies 1-2.  At the start of step 2s+1 a wave waits for its
// copies of stage s+1 (only x of stage s+2 may still be in flight), then
// barrier.  The fragments of step k+1 are read during step k, so a slot is
// free once the barrier at the start of the last step of its stage has
// passed.  NC = 0: a wave that copies nothing (same barriers).
template <typename T, int NC>
__device__ __forceinline__ void mainloop_256(char* smem, const T* __restrict__ X, const T* __restrict__ Wt, int M,
                                             int N, int K, int m0, int n0,
                                             f32x4 (&acc)[BigTile::NB][BigTile::MB], int wave, int lane, int rev,
                                             uint64_t& t_ready) {
  constexpr int NB = BigTile::NB, MB = BigTile::MB, WTM = BigTile::WTM, WTN = BigTile::WTN, WGN = BigTile::WGN;
  constexpr int SLOT = 256 * ROWB;        // one operand's stage: 32 KB
  constexpr int NCA = NC > 0 ? NC : 1;
  constexpr int WR = NC * 8;              // stage rows copied by one wave (64)
  constexpr int CG = 2;                   // n blocks of a step that issue its copies
  constexpr int CPG = NC / CG;            // copies per such n block
  constexpr int UNR = 12;                 // steps per loop iteration: 6 stages, a multiple of 3 and 2
  static_assert(MB == 8 && NB == 4, "the step's schedule assumes 8 x 4 result blocks per wave");
  static_assert(NC == 0 || (NC % CG == 0 && WR * 4 == 256), "four copying waves cover the 256 stage rows");
  const uint32_t rowbytes = (uint32_t)K * sizeof(T);
  const u32x4 rx = make_rsrc(X, (uint32_t)M * rowbytes);
  const u32x4 rw = make_rsrc(Wt, (uint32_t)N * rowbytes);
  // copy j of this wave covers slot rows wave*WR + 8j .. +7; lane i writes row
  // +i/8, 16-byte slot i%8, and loads global chunk slot ^ swizzle(row)
  uint32_t vx[NCA], vw[NCA];
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    const int srow = wave * WR + j * 8 + lane / 8;
    const int chunk = (lane % 8) ^ row_swizzle(srow);
    int gx = m0 + srow;
    gx = gx < M ? gx : M - 1;   // rows past the edge re-read the last row (never stored)
    int gw = n0 + srow;
    gw = gw < N ? gw : N - 1;
    vx[j] = (uint32_t)gx * rowbytes + chunk * 16;
    vw[j] = (uint32_t)gw * rowbytes + chunk * 16;
  }
  const uint32_t cbase = (uint32_t)(uintptr_t)smem + wave * WR * ROWB;   // this wave's first slot row

#define NSW_XSLOT(s) (((s) % 3) * SLOT)
#define NSW_WSLOT(s) ((3 + (s) % 2) * SLOT)
// copy j of stage st (k bytes st*ROWB ..) into the slot of stage sl (sl == st
// modulo 6; sl is a compile-time constant)
// k offset of stage st: stages walked from the last one when rev_ is set
#define NSW_KOFF(st) ((uint32_t)(rev_ ? (nst - 1 - (st)) : (st)) * ROWB)
#define NSW_COPY_X(sl, st, j) dma16(rx, cbase + NSW_XSLOT(sl) + (j) * 1024, vx[j], NSW_KOFF(st))
#define NSW_COPY_W(sl, st, j) dma16(rw, cbase + NSW_WSLOT(sl) + (j) * 1024, vw[j], NSW_KOFF(st))

  const int nk = K / (STEPB / (int)sizeof(T));   // MFMA steps
  // stages; with an odd step count the last stage holds one step's k (its
  // second half is copied -- the next row's first bytes, or zeros past the
  // end of the operand -- and never read by an MFMA)
  const int nst = (nk + 1) / 2;
  // serpentine k: a tile of an odd round of its XCD walks the stages from
  // the last one, so that it starts on the k slabs the tiles before it on
  // the XCD finished with, still in L2 (odd step counts keep the half
  // stage last: forward)
  const bool rev_ = rev && (nk & 1) == 0;
  // prologue: x0 w0 x1 w1, then wait for x0 and w0 (step 0 issues x2)
#pragma unroll
  for (int j = 0; j < NC; ++j) NSW_COPY_X(0, 0, j);
#pragma unroll
  for (int j = 0; j < NC; ++j) NSW_COPY_W(0, 0, j);
  if (nst > 1) {
#pragma unroll
    for (int j = 0; j < NC; ++j) NSW_COPY_X(1, 1, j);
#pragma unroll
    for (int j = 0; j < NC; ++j) NSW_COPY_W(1, 1, j);
    NSW_WAIT_VMCNT(2 * NC);
  } else {
    NSW_WAIT_VMCNT(0);
  }
  wg_barrier();
  NSW_STAMP(t_ready);

  const int frow = lane & 15, fg = lane >> 4;
  const int wrow = (wave % WGN) * WTN + frow;  // w rows of this wave (A operand)
  const int xrow = (wave / WGN) * WTM + frow;  // x rows of this wave (B operand)
  u32x4 fa[2][NB], fb[2][MB];
#pragma unroll
  for (int i = 0; i < NB; ++i) fa[0][i] = lds_frag(smem + NSW_WSLOT(0), wrow + i * 16, fg);
#pragma unroll
  for (int i = 0; i < MB; ++i) fb[0][i] = lds_frag(smem + NSW_XSLOT(0), xrow + i * 16, fg);

  // step k = kt + U of stage st = k/2; kt is a multiple of UNR, so the slots
  // of the stages touched by step U are compile-time constants.  Step k
  // copies stage st + 2 (x in its first step, w in its second) with no
  // condition: uniform branches around the copies cost ~7% of the loop.  Past
  // the last stage these copies re-read the last stage (L2-resident) into
  // slots nothing reads: x into the slot of stage st - 1,
  // w into the slot of stage st, which the barrier at the start of the step
  // has freed, except in the last step (no barrier): its w copies go to the
  // x slot of stage st + 1, unused.  The epilogue drains them before it
  // writes LDS.
#define NSW_STEP256(U)                                                                         \
  {                                                                                            \
    const int k = kt + U;                                                                      \
    if (k < nk) {                                                                              \
      constexpr int sub_ = (U) % 2, su_ = (U) / 2;                                             \
      constexpr int nsub_ = ((U) + 1) % 2, nsu_ = ((U) + 1) / 2;                               \
      const int st = k >> 1;                                                                   \
      if (sub_ == 1 && k + 1 < nk) {                                                           \
        NSW_WAIT_VMCNT(NC);                                                                    \
        NSW_WAIT_LGKMCNT0();                                                                   \
        wg_barrier();                                                                          \
      }                                                                                        \
      const uint32_t wdst_ = cbase + (k + 1 < nk ? NSW_WSLOT(su_ + 2) : NSW_XSLOT(su_ + 1));    \
      const int cst_ = st + 2 < nst ? st + 2 : nst - 1;   /* past the end: the last stage, in L2 */ \
      /* n-block-major: the first MFMAs of a step need only its first weight  */             \
      /* fragment.  Per n block: the copies (first CG blocks), MB/NB next-step */            \
      /* x fragments, MB MFMAs, then the next step's weight fragment nb into   */            \
      /* the registers the MFMAs have just released (two sets of x fragments, */             \
      /* one of w)                                                             */            \
      _Pragma("unroll") for (int nb = 0; nb < NB; ++nb) {                                      \
        if (nb < CG) {                                                                         \
          _Pragma("unroll") for (int c_ = 0; c_ < CPG; ++c_) {                                 \
            const int j_ = nb * CPG + c_;                                                      \
            if (sub_ == 1) dma16(rw, wdst_ + j_ * 1024, vw[j_], NSW_KOFF(cst_));                \
            else NSW_COPY_X(su_ + 2, cst_, j_);                                                \
          }                                                                                    \
        }                                                                                      \
        /* unconditional: after the last step these read stale slots (unused); a  */         \
        /* conditional read would make the wait-count pass drain all LDS reads   */         \
        _Pragma("unroll") for (int q = 0; q < MB / NB; ++q) {                                  \
          const int mq = nb * (MB / NB) + q;                                                   \
          fb[((U) + 1) & 1][mq] = lds_frag(smem + NSW_XSLOT(nsu_), xrow + mq * 16, nsub_ * 4 + fg); \
        }                                                                                      \
        _Pragma("unroll") for (int mb = 0; mb < MB; ++mb)                                      \
          mfma_bf16(acc[nb][mb], __builtin_bit_cast(bf16x8, fa[(U) & 1][nb]), __builtin_bit_cast(bf16x8, fb[(U) & 1][mb]));                        \
        fa[((U) + 1) & 1][nb] = lds_frag(smem + NSW_WSLOT(nsu_), wrow + nb * 16, nsub_ * 4 + fg); \
        /* the group's three fragment reads spread over its MFMAs: 1, 2 MFMAs, 1, */            \
        /* 3 MFMAs, 1, 3 MFMAs                                                    */            \
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                                     \
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);\
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                                     \
        __builtin_amdgcn_sched_group_barrier(0x008, 3, 0);\
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                                     \
        __builtin_amdgcn_sched_group_barrier(0x008, 3, 0);\
      }                                                                                        \
    }                                                                                          \
  }

  for (int kt = 0; kt < nk; kt += UNR) {
    NSW_STEP256(0) NSW_STEP256(1) NSW_STEP256(2) NSW_STEP256(3)
    NSW_STEP256(4) NSW_STEP256(5) NSW_STEP256(6) NSW_STEP256(7)
    NSW_STEP256(8) NSW_STEP256(9) NSW_STEP256(10) NSW_STEP256(11)
  }
#undef NSW_STEP256
#undef NSW_COPY_X
#undef NSW_KOFF
#undef NSW_COPY_W
#undef NSW_XSLOT
#undef NSW_WSLOT
}

// An fp32 value as the sum of three bf16: h = bf16(x), m = bf16(x - h),
// l = bf16(x - h - m), each difference exact.  h + m + l holds 24 significant
// bits, all of x's.
struct Split3 { bf16x8 h, m, l; };
__device__ __forceinline__ Split3 split3(const u32x4& a, const u32x4& b) {
  u32x4 h, m, l;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const f32x2 x = __builtin_bit_cast(f32x2, e < 2 ? uint2{a[2 * e], a[2 * e + 1]} : uint2{b[2 * e - 4], b[2 * e - 3]});
    // v_cvt_pk_bf16_f32 on pairs; the parts are widened back with shift and mask
    h[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(x, bf16x2));
    const f32x2 r = {x[0] - __builtin_bit_cast(float, h[e] << 16), x[1] - __builtin_bit_cast(float, h[e] & 0xffff0000u)};
    m[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, bf16x2));
    const f32x2 t = {r[0] - __builtin_bit_cast(float, m[e] << 16), r[1] - __builtin_bit_cast(float, m[e] & 0xffff0000u)};
    l[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(t, bf16x2));
  }
  return {__builtin_bit_cast(bf16x8, h), __builtin_bit_cast(bf16x8, m), __builtin_bit_cast(bf16x8, l)};
}

// Eight fp32 values times a power of two as the sums of two fp16: h = fp16(x s),
// l = fp16(x s - h), the difference exact.  h + l is within 2^-23 of |x s|, or
// 2^-25 where that is larger, up to |x s| = SPLIT2_MAX.
constexpr float SPLIT2_MAX = 65504.f;
__device__ __forceinline__ void split2(const f32x4& a, const f32x4& b, float sc, u32x4& h, u32x4& l) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float x0 = e < 2 ? a[2 * e] : b[2 * e - 4], x1 = e < 2 ? a[2 * e + 1] : b[2 * e - 3];
    const f16x2 hp = __builtin_convertvector((f32x2{x0 * sc, x1 * sc}), f16x2);
    h[e] = __builtin_bit_cast(uint32_t, hp);
    l[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{__builtin_fmaf(x0, sc, -(float)hp[0]),
                                                                       __builtin_fmaf(x1, sc, -(float)hp[1])}), f16x2));
  }
}

// Lanes that hold a magnitude |x s| below lo or above SPLIT2_MAX (NaN does not
// count).  The three-input forms as such: fminf and fmaxf put a canonicalising
// instruction before each value and cost 20% of the GEMM's time.
__device__ __forceinline__ uint64_t split2_outside(const f32x4& a, const f32x4& b, float sc, float lo) {
  float mn = fabsf(a[0]), mx = mn;
  auto min3 = [&](float x, float y) { asm("v_min3_f32 %0, |%1|, |%2|, %0" : "+v"(mn) : "v"(x), "v"(y)); };
  auto max3 = [&](float x, float y) { asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(mx) : "v"(x), "v"(y)); };
  min3(a[1], a[2]);
  max3(a[1], a[2]);
  min3(a[3], b[0]);
  max3(a[3], b[0]);
  min3(b[1], b[2]);
  max3(b[1], b[2]);
  min3(b[3], b[3]);
  max3(b[3], b[3]);
  return __ballot(mn * sc < lo) | __ballot(mx * sc > SPLIT2_MAX);
}

// Whether two parts hold x at scale s.
__device__ __forceinline__ bool split2_holds(float x, float s, float lo) {
  const float m = fabsf(x * s);
  return x == 0.f || (m >= lo && m <= SPLIT2_MAX);
}

// Scale of a row from the eight values that each lane of its quad holds: takes
// the second smallest of the four lanes' largest magnitudes to [2^11, 2^12), which
// leaves 2^4 above it and 2^15 to 2^17 below.  (Units listed of 256 rows, normal K
// = 1024 / GELU of normal values K = 4096 / a Student t of 3 degrees K = 1024:
// smallest to 2^12 1 / 961 / 155, to 2^11 1 / 11 / 24; second smallest to 2^11 2 /
// 9 / 6, to 2^10 7 / 21 / 8; largest to 2^10 9 / 35 / 14, and that follows
// outliers.)  0 while every value is zero.
__device__ __forceinline__ float split2_scale(const f32x4& a, const f32x4& b) {
  float m = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) m = fmaxf(m, fmaxf(fabsf(a[e]), fabsf(b[e])));
  m = quad_second_min(m == 0.f ? INFINITY : m);
  int ex = (int)(__builtin_bit_cast(uint32_t, m) >> 23) - 127;   // 2^ex <= m < 2^(ex + 1)
  ex = ex < -115 ? -115 : ex;
  return m == INFINITY ? 0.f : __builtin_bit_cast(float, (uint32_t)(11 - ex + 127) << 23);
}

// acc += w x of one block from the operands' three parts, smallest products
// first, and the same for the NB blocks of a row block (independent
// accumulators between dependent ones).
__device__ __forceinline__ void mul_parts(f32x4& acc, const Split3& w, const Split3& x) {
  mfma_bf16(acc, w.l, x.h);
  mfma_bf16(acc, w.h, x.l);
  mfma_bf16(acc, w.m, x.m);
  mfma_bf16(acc, w.m, x.h);
  mfma_bf16(acc, w.h, x.m);
  mfma_bf16(acc, w.h, x.h);
}
template <int NB, int MB>
__device__ __forceinline__ void mul_parts4(f32x4 (&acc)[NB][MB], int mb, const Split3 (&w)[NB], const Split3& x) {
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) mfma_bf16(acc[nb][mb], w[nb].l, x.h);
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) mfma_bf16(acc[nb][mb], w[nb].h, x.l);
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) mfma_bf16(acc[nb][mb], w[nb].m, x.m);
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) mfma_bf16(acc[nb][mb], w[nb].m, x.h);
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) mfma_bf16(acc[nb][mb], w[nb].h, x.m);
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) mfma_bf16(acc[nb][mb], w[nb].h, x.h);
}

// Operand copies of the ring main loops: a stage is 128 bytes of k of BM x rows
// and BN w rows.  Copy j of a wave covers stage rows (wave * CX + j) * 8 .. +7
// of x (j < CX) or of w; lane i writes row +i/8, 16-byte slot i%8, and loads
// global chunk slot ^ swizzle(row).  Rows past the edge re-read the last row
// (never stored).
template <typename T, class TC> struct StageCopy {
  static constexpr int NW = TC::NW;
  static constexpr int CX = TC::BM / 8 / NW, CW = TC::BN / 8 / NW;   // 1 KB copies per wave and stage
  static constexpr int NC = CX + CW;
  static_assert(CX * NW * 8 == TC::BM && CW * NW * 8 == TC::BN, "copies split evenly over the waves");
  u32x4 rx, rw;
  uint32_t v[NC], cx, cw;
  int wave, lane, nk, nst;   // nst: stages; an odd step count leaves half of the last one unused

  __device__ __forceinline__ void init(const char* smem, const T* X, const T* Wt, int M, int N, int K, int m0, int n0,
                                       int wave_, int lane_) {
    wave = wave_;
    lane = lane_;
    const uint32_t rowbytes = (uint32_t)K * sizeof(T);
    rx = make_rsrc(X, (uint32_t)M * rowbytes);
    rw = make_rsrc(Wt, (uint32_t)N * rowbytes);
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const int r = row(j) + lane / 8;
      const int g = j < CX ? (m0 + r < M ? m0 + r : M - 1) : (n0 + r < N ? n0 + r : N - 1);
      v[j] = (uint32_t)g * rowbytes + (uint32_t)((lane % 8) ^ row_swizzle(r)) * 16u;
    }
    cx = (uint32_t)(uintptr_t)smem + (uint32_t)(wave * CX * 1024);
    cw = (uint32_t)(uintptr_t)smem + (uint32_t)(TC::BM * ROWB + wave * CW * 1024);
    nk = K / (STEPB / (int)sizeof(T));
    nst = (nk + 1) / 2;
  }
  // first row of copy j within its operand's part of the stage
  __device__ __forceinline__ int row(int j) const { return j < CX ? (wave * CX + j) * 8 : (wave * CW + j - CX) * 8; }
  // copies [lo, hi) of stage s into a slot.  fp32: the unused half of the last
  // stage reads past the end of the operands (the range check returns zeros),
  // so that it adds nothing to the step, which takes whole stages.
  __device__ __forceinline__ void copy(int s, int slot, int lo, int hi) const {
    const uint32_t so = (uint32_t)slot * (uint32_t)TC::SLOT;
    const bool half = sizeof(T) == 4 && (nk & 1) != 0 && s == nst - 1;
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      if (j < lo || j >= hi) continue;
      const int chunk = (lane % 8) ^ row_swizzle(row(j) + lane / 8);
      dma16(j < CX ? rx : rw, (j < CX ? cx + j * 1024u : cw + (j - CX) * 1024u) + so,
            half && chunk >= 4 ? 0x80000000u : v[j], (uint32_t)s * ROWB);
    }
  }
};

// bf16 main loop with a ring of NST stages, one barrier per stage: at the top
// of stage s a wave waits for its copies of stage s, and past the barrier
// (every wave's copies have landed, and every wave is done reading stage s -
// 1) it issues the copies of stage s + NST - 1 into the slot of stage s - 1.
template <class TC>
__device__ __forceinline__ void mainloop_ring(char* smem, const bf16* __restrict__ X, const bf16* __restrict__ Wt, int M,
                                              int N, int K, int m0, int n0, f32x4 (&acc)[TC::NB][TC::MB], int wave,
                                              int lane) {
  constexpr int NB = TC::NB, MB = TC::MB, NST = TC::NST;
  using Copy = StageCopy<bf16, TC>;
  Copy cp;
  cp.init(smem, X, Wt, M, N, K, m0, n0, wave, lane);
  const int nst = cp.nst;
#pragma unroll
  for (int s = 0; s < NST - 1; ++s)
    if (s < nst) cp.copy(s, s, 0, Copy::NC);
  const int frow = lane & 15, fg = lane >> 4;
  const int xrow = (wave / TC::WGN) * TC::WTM + frow;             // x rows of this wave (B operand)
  const int wrow = TC::BM + (wave % TC::WGN) * TC::WTN + frow;    // w rows of this wave (A operand)
  int slot = 0;
  for (int s = 0; s < nst; ++s) {
    // copies of the up to NST - 2 stages after s may stay in flight
    if (nst - 1 - s >= NST - 2) NSW_WAIT_VMCNT((NST - 2) * Copy::NC);
    else NSW_WAIT_VMCNT(0);
    wg_barrier();
    if (s + NST - 1 < nst) cp.copy(s + NST - 1, slot == 0 ? NST - 1 : slot - 1, 0, Copy::NC);
    const char* st = smem + slot * TC::SLOT;
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      if (sub == 1 && (cp.nk & 1) != 0 && s == nst - 1) break;   // the unused half of the last stage
      bf16x8 fa[NB];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) fa[nb] = __builtin_bit_cast(bf16x8, lds_frag(st, wrow + nb * 16, 4 * sub + fg));
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        const bf16x8 fb = __builtin_bit_cast(bf16x8, lds_frag(st, xrow + mb * 16, 4 * sub + fg));
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) mfma_bf16(acc[nb][mb], fa[nb], fb);
      }
    }
    slot = slot + 1 == NST ? 0 : slot + 1;
  }
}

// Units (16 rows x the 32 k of a stage) with a value that two fp16 parts do not
// hold (mainloop_split2).  Rows count the tile's x rows, then its w rows.  The list
// takes three quarters of a stage's units, so that it does not fit the first stage
// of a tile that has such values everywhere (with all 32 of a 256 x 256 tile listed
// and added, that tile took 2500 us for 64800 x 3072 x 1024 instead of 1880).
template <class TC> constexpr int split2_list = (TC::BM + TC::BN) / 16 * 3 / 4;
constexpr int SPLIT2_LIST = split2_list<BigTile>;
struct Split2List {
  int n;                  // units found; those past split2_list are not listed
  int stop;               // first stage with a unit that is not listed
  int row[SPLIT2_LIST];   // first row; SPLIT2_ONE + the row of a single small value
  int k[SPLIT2_LIST];
};
constexpr int SPLIT2_ONE = 1 << 16;

// Single small values below k end, whose parts are in the sums: each is at most
// 2^-25 short, so a result of its row at most 2^-25 SPLIT2_MAX < 2^-9 (all scaled).
// Returns the entries (bits) with a result of this wave that is not 2^20 times what
// the row's small values may take from it; what their parts are short of is to be
// added (normal rows, K = 1024: about 4 entries in 1000).  Results
// below 4 become NaN, which redo_nonfinite forms again: a product of a subnormal part
// takes part in the instruction's alignment as if the part were 2^-14, which may
// take 2^-22 from the others'.  Rows of x or of w that are zero throughout (sh:
// exponents of the rows' scales, 127 there) are left alone.
template <class TC>
__device__ __forceinline__ uint32_t check_small(const Split2List& list, const int* sh, int end,
                                                f32x4 (&acc)[TC::NB][TC::MB], int wave, int lane) {
  constexpr int NB = TC::NB, MB = TC::MB;
  static_assert(SPLIT2_LIST <= 32, "an entry is a bit");
  const int frow = lane & 15, fg = lane >> 4;
  const int n = __builtin_amdgcn_readfirstlane(list.n < split2_list<TC> ? list.n : split2_list<TC>);
  uint32_t add = 0;
#pragma unroll 1
  for (int i = 0; i < n; ++i) {
    int row = __builtin_amdgcn_readfirstlane(list.row[i]);
    if (row < SPLIT2_ONE || __builtin_amdgcn_readfirstlane(list.k[i]) >= end) continue;
    const float least = 0x1p11f * (float)__popcll(__ballot(lane < n && list.row[lane < n ? lane : 0] == row));
    row -= SPLIT2_ONE;
    const bool isx = row < TC::BM;
    const int r = isx ? row - (wave / TC::WGN) * TC::WTM : row - TC::BM - (wave % TC::WGN) * TC::WTN;   // of this wave
    if (r < 0 || r >= (isx ? TC::WTM : TC::WTN)) continue;
    const bool mine = isx ? frow == (r & 15) : fg == ((r >> 2) & 3);
    bool low = false;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        if ((isx ? mb : nb) != r >> 4) continue;
        const int xr = (wave / TC::WGN) * TC::WTM + mb * 16 + frow, wr = TC::BM + (wave % TC::WGN) * TC::WTN + nb * 16 + 4 * fg;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const float m = fabsf(acc[nb][mb][c]);
          if (mine && (isx || c == (r & 3)) && m < least && sh[xr] != 127 && sh[wr + c] != 127) {
            low = true;
            if (m < 4.f) acc[nb][mb][c] = __builtin_nanf("");
          }
        }
      }
    if (__ballot(low) != 0) add |= 1u << i;
  }
  return add;
}

// What the parts of a value outside the window are short of at scale s: all of it
// where it was given none (not small), else what they round away.
__device__ __forceinline__ float split2_rest(float x, float s, bool small) {
  const float v = x * s;
  if (!small || fabsf(v) <= 0x1p-25f) return x;
  const _Float16 h = (_Float16)v;
  const float d = v - (float)h;
  return __builtin_amdgcn_ldexpf(d - (float)(_Float16)d, 127 - (int)(__builtin_bit_cast(uint32_t, s) >> 23));
}

// What the parts of the listed units below k end are short of (of single small
// values: those in `small`), times the other operand, with the fp32 matrix
// instruction.  A pair of two values without parts counts once, for the unit of x;
// else the other operand's values count whole.  sh: exponents of the rows' scales.
// The sums of a unit pass through LDS (buf, a KB a block), so that they are formed
// in one rolled loop: added to the accumulators where they are formed, the
// accumulators spilled.  2 us a unit of x and 5 us a unit of w of a 256 x 256 tile,
// a quarter of that for the single small values that need nothing.
template <class TC>
__device__ __forceinline__ void add_outside(const Split2List& list, const int* sh, char* buf, const float* __restrict__ X,
                                            const float* __restrict__ Wt, int M, int N, int K, int m0, int n0, int end,
                                            float lo, uint32_t small, f32x4 (&acc)[TC::NB][TC::MB], int wave, int lane) {
  constexpr int NB = TC::NB, MB = TC::MB;
  const int frow = lane & 15, fg = lane >> 4;
  const int xw = (wave / TC::WGN) * TC::WTM, ww = (wave % TC::WGN) * TC::WTN;   // this wave's first x and w rows
  const int n = __builtin_amdgcn_readfirstlane(list.n < split2_list<TC> ? list.n : split2_list<TC>);
  // lane i has entry i and its place in the order of k and row: the order of the
  // list is the waves', and sums are to repeat bit for bit
  const int lrow = list.row[lane < n ? lane : 0], lk = list.k[lane < n ? lane : 0];
  int place = 0;
  for (int i = 0; i < n; ++i) {
    const int r = __builtin_amdgcn_readlane(lrow, i), k = __builtin_amdgcn_readlane(lk, i);
    place += k < lk || (k == lk && r < lrow);
  }
#pragma unroll 1
  for (int t = 0; t < n; ++t) {
    const int i = __builtin_ctzll(__ballot(lane < n && place == t));
    int row = __builtin_amdgcn_readlane(lrow, i);
    const int k = __builtin_amdgcn_readlane(lk, i);
    const bool one = row >= SPLIT2_ONE;
    row &= SPLIT2_ONE - 1;
    const bool isx = row < TC::BM;
    const int blk = (isx ? row - xw : row - TC::BM - ww) >> 4;      // this wave's row block
    if (k >= end || (one && (small >> i & 1) == 0) || blk < 0 || blk >= (isx ? MB : NB)) continue;
    f32x4* sum = reinterpret_cast<f32x4*>(buf) + wave * (MB > NB ? MB : NB) * 64 + lane;
    // lane (i, g): k 4g..4g+3 and 16+4g..+3 of row i of a block (the second half
    // of the last stage may lie past K: zero)
    auto load = [&](bool ofx, int b, f32x4 (&v)[2]) {
      const int g = ofx ? m0 + xw + b * 16 + frow : n0 + ww + b * 16 + frow, rows = ofx ? M : N;
      const float* p = (ofx ? X : Wt) + (int64_t)(g < rows ? g : rows - 1) * K + k + 4 * fg;
      v[0] = *reinterpret_cast<const f32x4*>(p);
      v[1] = k + 16 < K ? *reinterpret_cast<const f32x4*>(p + 16) : f32x4{0.f, 0.f, 0.f, 0.f};
    };
    auto scale = [&](bool ofx, int b) {
      return __builtin_amdgcn_ldexpf(1.f, -sh[(ofx ? xw : TC::BM + ww) + b * 16 + frow]);
    };
    constexpr int G = MB < NB ? MB : NB;      // blocks of the other operand whose loads are in flight together
    f32x4 u[2];
    load(isx, blk, u);
    const float us = scale(isx, blk);
#pragma unroll 1
    for (int b = 0; b < (isx ? NB : MB); b += G) {
      f32x4 o[G][2];
#pragma unroll
      for (int j = 0; j < G; ++j) load(!isx, b + j, o[j]);
#pragma unroll
      for (int j = 0; j < G; ++j) {
        const float os = scale(!isx, b + j);
        // the other unit may have values without parts itself
        const int orow = isx ? TC::BM + ww + (b + j) * 16 : xw + (b + j) * 16;
        const bool both = (one || !isx) && __ballot(lane < n && lrow == orow && lk == k) != 0;
        f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          float r = u[e >> 2][e & 3], q = o[j][e >> 2][e & 3];
          r = split2_holds(r, us, lo) ? 0.f : split2_rest(r, us, one);
          if (both && !split2_holds(q, os, lo)) q = 0.f;
          c = __builtin_amdgcn_mfma_f32_16x16x4f32(isx ? q : r, isx ? r : q, c, 0, 0, 0);
        }
        sum[(b + j) * 64] = c;
      }
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
        if ((isx ? mb : nb) == blk) acc[nb][mb] += sum[(isx ? nb : mb) * 64];
  }
}

// fp32 main loop on two fp16 parts of each operand (rows scaled by powers of
// two), three products.  A stage is 32 k: one step of the 16-bit matrix
// instructions, lane group g taking k 4g..4g+3 and 16+4g..+3 of both operands.
//
// VALU work takes issue time from the matrix instructions here (measured: 7.2
// ns an MFMA alone, 9.1 with two subtractions between, 12.5 with two
// v_fma_mixlo_f16), so each value is split once a workgroup, not once in every
// wave that reads it: the wave that copied 16 stage rows splits them in place,
// the h parts into the chunk of k 4c.. and the l parts into that of 16+4c...
//
// A ring of two slots.  In stage s the wave splits its rows of stage s + 1 under
// the MFMAs before row block BARB; the stage's one barrier stands there, once
// every fragment of the stage is in registers: past it the next stage's first
// fragments are read, and the copies of stage s + 2 start into the slot just
// read.  Issued in one go the copies hold every wave for the ~1000 cycles that
// the CU's address path takes for 64 KB, so they are spread, and they carry no
// condition (past the end they re-read the last stage into a slot whose values
// are not used).
//
// Range.  Two parts hold a scaled magnitude between lo and SPLIT2_MAX to 2^-25 /
// lo of itself or better, and zero.  Every value is looked at before it is split.
// The unit of one outside goes on a list.  A single small value keeps its parts;
// the results of its row are looked at in the end, and what the parts are short of
// is added where it matters (check_small, add_outside).  Otherwise the values
// outside get zero parts and their products are added in the end.  A product keeps
// within (K / 8 + 4) 2^-24 of itself whatever else its rows hold, a quarter of what
// K fp32 additions may lose: lo = 8 / K costs each of the two values K / 16 2^-24,
// and leaving out the product of the l parts 4 2^-24.  lo is no lower than 2^-6, so
// that a value is never further off than 2^-19.  Rows of normal values put about 5 K
// / 1024 units of a 256 x 256 tile on the list, nearly all with one small value.  A
// tile whose list is full leaves the loop before the stage that did not fit; the
// caller goes on from that stage (the return value) on three parts.
//
// A row's scale is set at its first stage that is not zero throughout
// (split2_scale; until then it is 0).
template <class TC>
__device__ __forceinline__ int mainloop_split2(char* smem, Split2List& list, const float* __restrict__ X,
                                               const float* __restrict__ Wt, int M, int N, int K, int m0, int n0,
                                               f32x4 (&acc)[TC::NB][TC::MB], int wave, int lane) {
  constexpr int NB = TC::NB, MB = TC::MB;
  constexpr int BARB = MB > 2 ? MB - 2 : 1;      // row block before which the barrier stands
  using Copy = StageCopy<float, TC>;
  constexpr int NC = Copy::NC, NU = NC / 2;      // copies, 16-row units to split
  constexpr int NC1 = NC * 3 / 4;                // copies issued past the barrier; the others in the next stage
  constexpr int SPLB = BARB > 2 ? 2 : BARB - 1;  // first row block with splits
  static_assert(TC::NST == 2, "a ring of two slots");
  static_assert(Copy::CX % 2 == 0 && Copy::CW % 2 == 0, "units of 16 rows of one operand");
  Copy cp;
  cp.init(smem, X, Wt, M, N, K, m0, n0, wave, lane);
  const int nst = cp.nst;
  const float lo = fmaxf(8.f / (float)K, 0x1p-6f);
  cp.copy(0, 0, 0, NC);
  cp.copy(nst > 1 ? 1 : 0, 1, 0, NC1);
  // this lane's row of a unit and its chunk pair (c, c + 4): any 16 lanes
  // cover four rows whose pairs lie in distinct banks
  const int li = lane >> 2, lc = lane & 3;
  const int urow = (li & 1) | ((li >> 1) & 1) << 3 | (li >> 2) << 1;
  const int uoff = urow * ROWB + (lc ^ row_swizzle(urow)) * 16;   // chunk c; chunk c + 4 is at ^ 64
  auto unit = [&](int u) { return (u < Copy::CX / 2 ? 0 : TC::BM * ROWB) + cp.row(2 * u) * ROWB + uoff; };
  float sc[NU];
  // looks at unit u of stage s: a, b stay what is to be split
  auto look = [&](int u, int s, f32x4& a, f32x4& b) {
    if (__builtin_expect(split2_outside(a, b, sc[u], lo) == 0, 1)) return;
    // a value outside the window, or a zero
    if (__ballot(sc[u] == 0.f) != 0) {
      const float t = split2_scale(a, b);
      if (sc[u] == 0.f) sc[u] = t;
    }
    const int row = (u < Copy::CX / 2 ? 0 : TC::BM) + cp.row(2 * u);
    const bool stored = u < Copy::CX / 2 ? m0 + row + urow < M : n0 + row + urow - TC::BM < N;   // not a repeated last row
    int count = 0;
    bool large = false;
    auto see = [&](float x) {
      count += !split2_holds(x, sc[u], lo);
      large |= !(fabsf(x * sc[u]) <= SPLIT2_MAX);
    };
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      see(a[e]);
      see(b[e]);
    }
    const uint64_t lanes = __ballot(count != 0 && stored);
    const bool one = __popcll(lanes) == 1 && __ballot(count > 1 || large) == 0;
    if (!one) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        a[e] = split2_holds(a[e], sc[u], lo) ? a[e] : 0.f;
        b[e] = split2_holds(b[e], sc[u], lo) ? b[e] : 0.f;
      }
    }
    if (lanes != 0 && s < nst && lane == (one ? __builtin_ctzll(lanes) : 0)) {
      const int i = __hip_atomic_fetch_add(&list.n, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      if (i < split2_list<TC>) {
        list.row[i] = one ? SPLIT2_ONE + row + urow : row;
        list.k[i] = s * 32;
      } else {
        __hip_atomic_fetch_min(&list.stop, s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    }
  };
  // the parts of unit u into its slot
  auto put = [&](int u, char* st, const f32x4& a, const f32x4& b) {
    u32x4 h, l;
    split2(a, b, sc[u], h, l);
    *reinterpret_cast<u32x4*>(st + unit(u)) = h;
    *reinterpret_cast<u32x4*>(st + (unit(u) ^ 64)) = l;
  };
  if (wave == 0 && lane == 0) {
    list.n = 0;
    list.stop = 0x7fffffff;
  }
  wg_barrier();        // the list is empty before any wave adds to it
  wait_copies<NC1>();
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    f32x4 a = *reinterpret_cast<const f32x4*>(smem + unit(u)), b = *reinterpret_cast<const f32x4*>(smem + (unit(u) ^ 64));
    sc[u] = split2_scale(a, b);
    look(u, 0, a, b);
    put(u, smem, a, b);
  }
  wg_barrier();
  const int frow = lane & 15, fg = lane >> 4;
  const int xrow = (wave / TC::WGN) * TC::WTM + frow;             // x rows of this wave (B operand)
  const int wrow = TC::BM + (wave % TC::WGN) * TC::WTN + frow;    // w rows of this wave (A operand)
  auto load = [&](const char* st, int row, f16x8 (&r)[2]) {
    r[0] = __builtin_bit_cast(f16x8, lds_frag(st, row, fg));
    r[1] = __builtin_bit_cast(f16x8, lds_frag(st, row, 4 + fg));
  };
  f16x8 ws[NB][2], wn[NB][2], xs[3][2];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) load(smem, wrow + nb * 16, ws[nb]);
  load(smem, xrow, xs[0]);
  load(smem, xrow + 16, xs[1]);
  // the first stage not to be run; a wave that is a stage ahead may have put a
  // later stage into list.stop by the time another reads it, never this one
  auto stopped = [&](int s) { return __builtin_amdgcn_readfirstlane(list.stop) <= s; };
  int s = 0;
  for (bool stop = stopped(0); s < nst && !stop; ++s) {
    char* st = smem + (s & 1) * TC::SLOT;
    char* sn = smem + ((s + 1) & 1) * TC::SLOT;
    // the rest of stage s + 1 here, most of stage s + 2 past the barrier
    const int c1 = s + 1 < nst ? s + 1 : nst - 1, c2 = s + 2 < nst ? s + 2 : nst - 1;
    cp.copy(c1, (s + 1) & 1, NC1, NC);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      if (mb == BARB) {
        wg_barrier();
        stop = stopped(s + 1);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) load(sn, wrow + nb * 16, wn[nb]);
      }
      if (mb >= BARB) {
        constexpr int L = MB - BARB;                 // row blocks past the barrier
        cp.copy(c2, s & 1, (mb - BARB) * NC1 / L, (mb - BARB + 1) * NC1 / L);
      }
      if (mb + 2 < MB) load(st, xrow + (mb + 2) * 16, xs[(mb + 2) % 3]);
      // the units of the next stage, split ahead of the barrier
      if (mb == SPLB) wait_copies();
      f32x4 ua[NU], ub[NU];
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        if (mb != SPLB + u * (BARB - SPLB) / NU) continue;
        ua[u] = *reinterpret_cast<const f32x4*>(sn + unit(u));
        ub[u] = *reinterpret_cast<const f32x4*>(sn + (unit(u) ^ 64));
      }
      const f16x8 (&x)[2] = xs[mb % 3];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) mfma_f16(acc[nb][mb], ws[nb][1], x[0]);
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        if (mb != SPLB + u * (BARB - SPLB) / NU) continue;
        look(u, s + 1, ua[u], ub[u]);
        put(u, sn, ua[u], ub[u]);
      }
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) mfma_f16(acc[nb][mb], ws[nb][0], x[1]);
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) mfma_f16(acc[nb][mb], ws[nb][0], x[0]);
    }
    load(sn, xrow, xs[0]);
    load(sn, xrow + 16, xs[1]);
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int i = 0; i < 2; ++i) ws[nb][i] = wn[nb][i];
  }
  wait_copies();       // those past the last stage
  wg_barrier();        // the ring is no longer read
  // scale back: the rows' exponents pass through LDS (a row without a scale is
  // zero throughout)
  int* sh = reinterpret_cast<int*>(smem);
#pragma unroll
  for (int u = 0; u < NU; ++u)
    if (lc == 0) sh[(u < Copy::CX / 2 ? 0 : TC::BM) + cp.row(2 * u) + urow] = 127 - (int)(__builtin_bit_cast(uint32_t, sc[u]) >> 23);
  wg_barrier();
  const uint32_t small = check_small<TC>(list, sh, s * 32, acc, wave, lane);
  int ex[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) ex[mb] = sh[xrow + mb * 16];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int4 ew = *reinterpret_cast<const int4*>(sh + TC::BM + (wave % TC::WGN) * TC::WTN + nb * 16 + 4 * fg);
    const int e[4] = {ew.x, ew.y, ew.z, ew.w};
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) acc[nb][mb][r] = __builtin_amdgcn_ldexpf(acc[nb][mb][r], e[r] + ex[mb]);
  }
  add_outside<TC>(list, sh, smem + 4096, X, Wt, M, N, K, m0, n0, s * 32, lo, small, acc, wave, lane);
  wg_barrier();        // the exponents are no longer read
  return s;
}

// fp32 main loop on three bf16 parts of each operand, which hold any fp32
// value: of the nine products the six of weight >= 2^-16, smallest first, and
// the three dropped are below 2^-24 of the product, as fp32's own rounding.
// For short K (gemm_kernel) and, from stage `first` on, tiles that two scaled fp16
// parts do not hold.
// Stages, barrier and copies as mainloop_split2, but the parts do not fit in
// place, so every wave splits the fragments it reads: w block nb + 1 under the
// MFMAs of (nb, mb 0), x block mb + 1 under those of block mb.
template <class TC>
__device__ __forceinline__ void mainloop_split3(char* smem, const float* __restrict__ X, const float* __restrict__ Wt,
                                                int M, int N, int K, int m0, int n0, f32x4 (&acc)[TC::NB][TC::MB],
                                                int wave, int lane, int first) {
  constexpr int NB = TC::NB, MB = TC::MB;
  constexpr int BARB = MB > 2 ? MB - 2 : 1;      // row block before which the barrier stands
  using Copy = StageCopy<float, TC>;
  constexpr int NC = Copy::NC, NC1 = NC / 2;     // copies issued past the barrier / in the next stage
  Copy cp;
  cp.init(smem, X, Wt, M, N, K, m0, n0, wave, lane);
  const int nst = cp.nst;
  if (first >= nst) return;
  cp.copy(first, 0, 0, NC);
  cp.copy(first + 1 < nst ? first + 1 : first, 1, 0, NC1);
  const int frow = lane & 15, fg = lane >> 4;
  const int xrow = (wave / TC::WGN) * TC::WTM + frow;             // x rows of this wave (B operand)
  const int wrow = TC::BM + (wave % TC::WGN) * TC::WTN + frow;    // w rows of this wave (A operand)
  NSW_WAIT_VMCNT(NC1);
  wg_barrier();
  auto load = [&](const char* st, int row, u32x4 (&r)[2]) {
    r[0] = lds_frag(st, row, fg);
    r[1] = lds_frag(st, row, 4 + fg);
  };
  u32x4 rw_[NB][2], rx_[2][2];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) load(smem, wrow + nb * 16, rw_[nb]);
  load(smem, xrow, rx_[0]);
  load(smem, xrow + 16, rx_[1]);
  Split3 ws[NB], xs = split3(rx_[0][0], rx_[0][1]), w0 = split3(rw_[0][0], rw_[0][1]), xn;
  for (int s = first; s < nst; ++s) {
    const int slot = (s - first) & 1;
    const char* st = smem + slot * TC::SLOT;
    const char* sn = smem + (slot ^ 1) * TC::SLOT;
    const int c1 = s + 1 < nst ? s + 1 : nst - 1, c2 = s + 2 < nst ? s + 2 : nst - 1;
    if (MB > 2) load(st, xrow + 32, rx_[0]);
    ws[0] = w0;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      cp.copy(c1, slot ^ 1, NC1 + nb * (NC - NC1) / NB, NC1 + (nb + 1) * (NC - NC1) / NB);
      mul_parts(acc[nb][0], ws[nb], xs);
      if (nb + 1 < NB) ws[nb + 1] = split3(rw_[nb + 1][0], rw_[nb + 1][1]);
      else xn = split3(rx_[1][0], rx_[1][1]);
#pragma unroll
      for (int q = 0; q < 6; ++q) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);
      }
    }
#pragma unroll
    for (int mb = 1; mb < MB; ++mb) {
      xs = xn;
      if (mb == BARB) {
        NSW_WAIT_VMCNT(0);
        wg_barrier();
      }
      if (mb >= BARB) {
        constexpr int L = MB - BARB;             // row blocks past the barrier
        cp.copy(c2, slot, (mb - BARB) * NC1 / L, (mb - BARB + 1) * NC1 / L);
      }
      if (mb + 2 < MB) load(st, xrow + (mb + 2) * 16, rx_[mb & 1]);
      if (mb == BARB) {
        load(sn, wrow, rw_[0]);
        load(sn, xrow, rx_[0]);
        if (MB == 2) load(sn, xrow + 16, rx_[1]);
      }
      if (mb == MB - 1) {
#pragma unroll
        for (int nb = 1; nb < NB; ++nb) load(sn, wrow + nb * 16, rw_[nb]);
        if (MB > 2) load(sn, xrow + 16, rx_[1]);
      }
      mul_parts4(acc, mb, ws, xs);
      if (mb + 1 < MB) xn = split3(rx_[(mb + 1) & 1][0], rx_[(mb + 1) & 1][1]);
      else {
        w0 = split3(rw_[0][0], rw_[0][1]);
        xn = split3(rx_[0][0], rx_[0][1]);
      }
#pragma unroll
      for (int q = 0; q < NB * 6; ++q) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
      }
    }
    xs = xn;
  }
  NSW_WAIT_VMCNT(0);   // the copies past the last stage
  wg_barrier();        // the ring is no longer read
}

// Whether one of the wave's results is not finite (the same on every lane).
template <class TC>
__device__ __forceinline__ bool any_nonfinite(const f32x4 (&acc)[TC::NB][TC::MB]) {
  float t = 0.f;
#pragma unroll
  for (int nb = 0; nb < TC::NB; ++nb)
#pragma unroll
    for (int mb = 0; mb < TC::MB; ++mb)
#pragma unroll
      for (int r = 0; r < 4; ++r) t = fmaf(acc[nb][mb][r], 0.f, t);   // NaN once a value is not finite
  return __ballot(!(t == 0.f)) != 0;
}

// fp32 results that are not finite are formed again with the fp32 matrix
// instruction: an infinite operand (or one that bf16 rounds to infinity, above
// 3.39e38) has no finite parts, so the split gives NaN where fp32 gives an
// infinity or a finite sum.  Only these results are replaced.  Operands straight
// from global memory; of a wave's 16 x 16 blocks those with such a result, a few at
// a time through LDS (buf, a KB each; with a loop for every block in the code, the
// loads could not run ahead).  On finite data no wave does.
template <class TC>
__device__ __forceinline__ void redo_nonfinite(char* buf, const float* __restrict__ X, const float* __restrict__ Wt, int M,
                                               int N, int K, int mw0, int nw0, f32x4 (&acc)[TC::NB][TC::MB], int wave,
                                               int lane) {
  constexpr int NB = TC::NB, MB = TC::MB, G = 4;
  static_assert(TC::NW * G * 1024 <= Stg<float, TC>::SMEM, "LDS layout");
  if (!any_nonfinite<TC>(acc)) return;
  const int frow = lane & 15, fg = lane >> 4;
  f32x4* c = reinterpret_cast<f32x4*>(buf) + wave * G * 64 + lane;
  uint32_t left = 0;     // blocks to be formed again: bits nb MB + mb
#pragma unroll
  for (int b = 0; b < NB * MB; ++b) {
    const f32x4 v = acc[b / MB][b % MB] * 0.f;        // NaN where a value is not finite
    if (__ballot(!((v[0] + v[1]) + (v[2] + v[3]) == 0.f)) != 0) left |= 1u << b;
  }
#pragma unroll 1
  while (left != 0) {
    uint32_t now = left;
#pragma unroll 1
    for (int g = 0; g < G && left != 0; ++g) {
      const int b = __builtin_ctz(left);
      left &= left - 1;
      const int n = nw0 + b / MB * 16 + frow, m = mw0 + b % MB * 16 + frow;
      const float* wp = Wt + (int64_t)(n < N ? n : N - 1) * K + 4 * fg;
      const float* xp = X + (int64_t)(m < M ? m : M - 1) * K + 4 * fg;
      f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
      for (int k = 0; k < K; k += 16) {
        const f32x4 w = *reinterpret_cast<const f32x4*>(wp + k);
        const f32x4 x = *reinterpret_cast<const f32x4*>(xp + k);
#pragma unroll
        for (int e = 0; e < 4; ++e) a = __builtin_amdgcn_mfma_f32_16x16x4f32(w[e], x[e], a, 0, 0, 0);
      }
      c[g * 64] = a;
    }
    now ^= left;
#pragma unroll
    for (int b = 0; b < NB * MB; ++b) {
      if (((now >> b) & 1) == 0) continue;
      const f32x4 a = c[__builtin_popcount(now & ((1u << b) - 1)) * 64];
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (!(acc[b / MB][b % MB][r] * 0.f == 0.f)) acc[b / MB][b % MB][r] = a[r];
    }
  }
}

// P consecutive values between LDS / registers / global memory, as one
// access where P * sizeof(V) is 2, 4, 8 or 16 bytes (16-byte pieces above).
template <typename V, int P>
__device__ __forceinline__ void copy_run(V* __restrict__ dst, const V* __restrict__ src) {
  constexpr int B = P * (int)sizeof(V);
  if constexpr (B >= 16) {
#pragma unroll
    for (int i = 0; i < B / 16; ++i) reinterpret_cast<u32x4*>(dst)[i] = reinterpret_cast<const u32x4*>(src)[i];
  } else if constexpr (B == 8) {
    *reinterpret_cast<uint2*>(dst) = *reinterpret_cast<const uint2*>(src);
  } else if constexpr (B == 4) {
    *reinterpret_cast<uint32_t*>(dst) = *reinterpret_cast<const uint32_t*>(src);
  } else {
    *reinterpret_cast<uint16_t*>(dst) = *reinterpret_cast<const uint16_t*>(src);
  }
}

// EPI_UNPATCH write-out of the staged rows [r0, r0 + S::ROWS) of a tile: the
// head layout of models/swin.py:286-299 (reshape [b, h, w, p, p, c], einsum
// nthwpqc -> ntchpwq) with the head's output columns permuted to c p^2 +
// dy p + dx (host side), so that a tile's BN columns are the whole p x p
// patches of BN / p^2 channels.  A thread keeps one staged row (a token:
// frame b, patch row py, patch column px) and walks the (channel, dy)
// pairs; per pair one LDS read of the p values dx = 0 .. p-1 and one store
// of p pixels into image row py p + dy.  Consecutive lanes hold consecutive
// tokens, so a store instruction covers consecutive p-pixel runs of one
// image row.  Values are rounded to T at staging, then widened to float for
// a float image (as the separate GEMM + unpatchify would).
template <typename T, class TC, int P>
__device__ __forceinline__ void unpatch_copy_out(const char* stg, const EpiArgs& ea, int M, int N, int r0, int n0,
                                                 int tid) {
  using S = Stg<T, TC>;
  constexpr int CPT = TC::BN / (P * P);               // channels per tile
  constexpr int TPR = TC::NW * 64 / S::ROWS;          // threads per staged row
  static_assert(CPT >= 1 && TPR >= 1, "whole patches per tile, a thread per row");
  const int tl = tid % S::ROWS;                       // staged row of this thread
  const int m = r0 + tl;
  if (m >= M) return;
  const int wq = ea.img_W / P, hw = (ea.img_H / P) * wq;
  const int b = m / hw, rr = m - b * hw, py = rr / wq, px = rr - py * wq;
  const int64_t HW = (int64_t)ea.img_H * ea.img_W;
  const int64_t pix0 = (int64_t)b * ea.img_bstride + (int64_t)(py * P) * ea.img_W + px * P;
  const int c0 = n0 / (P * P);
  const T* row = reinterpret_cast<const T*>(stg + tl * S::STRIDE);
  for (int cd = tid / S::ROWS; cd < CPT * P; cd += TPR) {
    const int cl = cd / P, dy = cd - cl * P;
    const int c = c0 + cl;
    if (c * P * P >= N) break;                        // columns past N: channels past C_out
    const T* src = row + cl * P * P + dy * P;
    const int64_t off = pix0 + c * HW + (int64_t)dy * ea.img_W;
    if (ea.img_f32 && sizeof(T) == 2) {
      T v[P];
      copy_run<T, P>(v, src);
      float f[P];
#pragma unroll
      for (int e = 0; e < P; ++e) f[e] = to_f32(v[e]);
      copy_run<float, P>(reinterpret_cast<float*>(ea.img) + off, f);
    } else {
      copy_run<T, P>(reinterpret_cast<T*>(ea.img) + off, src);
    }
  }
}

template <typename T, int EPI, int PRE, class TC>
__global__ __launch_bounds__(TC::NW * 64, TC::MINW) void gemm_kernel(const T* __restrict__ X, const T* __restrict__ Wt,
                                                                 T* __restrict__ Y, int M, int N, int K, EpiArgs ea) {
  constexpr int BM = TC::BM, BN = TC::BN, WTM = TC::WTM, WTN = TC::WTN, MB = TC::MB, NB = TC::NB, NW = TC::NW;
  constexpr int WGM = TC::WGM, WGN = TC::WGN;
  using S = Stg<T, TC>;
  constexpr int PRM_NW = S::PRM_NW, PRM_RS = S::PRM_RS;
  // the operand ring during the k loop, the output staging area in the
  // epilogue
  __shared__ __attribute__((aligned(1024))) char smem[S::SMEM];

  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int wm = wave / WGN, wn = wave % WGN;

  const int MT = (M + BM - 1) / BM, NT = (N + BN - 1) / BN;
  // Tiles of one XCD run in groups of GROUP_M row blocks x all column blocks,
  // column-major inside the group, so that the tiles in flight on an XCD
  // share both their row panels and their weight panels in its L2.
  // (ea.group_m 256-row blocks when set: 4 for the QKV projection and 16 for
  // proj, each measured 1.5-3% faster there; fc1 is fastest at 8)
  const int GM = (ea.group_m > 0 ? ea.group_m : GROUP_M) * (256 / BM);
  const int tile = xcd_remap(blockIdx.x, MT * NT);
  const int group = tile / (GM * NT);
  const int gm0 = group * GM;
  const int gsz = MT - gm0 < GM ? MT - gm0 : GM;
  const int tin = tile - group * GM * NT;
  const int mt = gm0 + tin % gsz, nt = tin / gsz;
  const int m0 = mt * BM, n0 = nt * BN;

  f32x4 acc[NB][MB];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < MB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // waves 0-3 copy the operands, waves 4-7 do not (see mainloop_256).  The
  // XCD-local workgroup index (blockIdx / 8) over the XCD's 32 CUs counts
  // the rounds of tiles on an XCD; odd rounds walk k backwards (serpentine:
  // 7-8% less L2 fetch on the K = 1024 GEMMs of config 2, 1-1.5% faster)
  const int rev = ((int)(blockIdx.x >> 3) / 32) & 1;
  uint64_t ts[5] = {0, 0, 0, 0, 0};   // phase stamps (NSW_GEMM_STAMPS builds only)
  NSW_STAMP(ts[0]);
  {
    const int lane0 = (int)threadIdx.x & 63;
    if constexpr (is_main256<T, TC>) {
      if (wave < 4) mainloop_256<T, 8>(smem, X, Wt, M, N, K, m0, n0, acc, wave, lane0, rev, ts[1]);
      else mainloop_256<T, 0>(smem, X, Wt, M, N, K, m0, n0, acc, wave, lane0, rev, ts[1]);
    } else if constexpr (sizeof(T) == 2) {
      mainloop_ring<TC>(smem, X, Wt, M, N, K, m0, n0, acc, wave, lane0);
    } else {
      // on two fp16 parts as long as they hold the tile's values, then on three
      // bf16 parts
      int stage = 0;
      if (K >= SPLIT2_MIN_K) {
        __shared__ Split2List list;
        stage = mainloop_split2<TC>(smem, list, X, Wt, M, N, K, m0, n0, acc, wave, lane0);
      }
      mainloop_split3<TC>(smem, X, Wt, M, N, K, m0, n0, acc, wave, lane0, stage);
      redo_nonfinite<TC>(smem, X, Wt, M, N, K, m0 + wm * WTM, n0 + wn * WTN, acc, wave, lane0);
    }
  }
  NSW_STAMP(ts[2]);
  // the lane's ids for the epilogue, from the lane counter and the (scalar)
  // wave id: kept live across the k loop they were spilled to scratch (2-5
  // VGPRs per instantiation; with this, none spill, bit-identical, time
  // unchanged).  Inline asm, or the compiler folds the counter back into the
  // work-item id and keeps that live.
  int lane;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane));
  const int tid = wave * 64 + lane;
  const int frow = lane & 15, fg = lane >> 4;

  // ---------------------------------------------------------------- epilogue
  // lane (frow, fg) of block (nb, mb) holds y[m0 + wm*WTM + mb*16 + frow]
  //                                          [n0 + wn*WTN + nb*16 + 4*fg + r]
  const int nw0 = n0 + wn * WTN;           // first column of this wave
  constexpr int HDQ = qkv_head_dim(EPI);
  // With the head norm or the row scale, the bias, norm weights and row
  // scales reach the lanes through LDS (one element per thread, parked there
  // once the operand ring is free): loaded straight into the fragment layout,
  // their 16+ small loads went out one at a time, each behind the previous
  // one, because the accumulators copied out of the AGPRs fill the VGPRs
  // here.  The bias-only epilogues load it directly (one batch).
  constexpr bool PLDS = HDQ > 0 || PRE == PRE_ROWSCALE;
  const T* bias = (const T*)ea.bias;
  float bv[NB][4];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int n = nw0 + nb * 16 + fg * 4;
#pragma unroll
    for (int r = 0; r < 4; ++r) bv[nb][r] = 0.f;
    if constexpr (EPI != EPI_NONE && EPI != EPI_UNPATCH && !PLDS)
      load4<T>(bias + (n < N ? n : 0), bv[nb]);   // straight-line: one batch
  }

  // per-head RMSNorm (QKV epilogue): a head is HDQ/16 consecutive 16-column
  // blocks inside one of the q / k / v regions (C % 16 == 0 and HDQ | C), so
  // whether a head is normalised is uniform across its lanes.  Head dims 4
  // and 8 put 4 / 2 heads in one 16-column block: a lane's 4 columns are a
  // whole head (4) or half of one, the other half in the lane 16 apart (8);
  // then the flags below are kept per block (NBH = 1, "heads" = blocks).
  constexpr int NBH = HDQ >= 16 ? HDQ / 16 : 1;  // blocks per head
  constexpr int HSP = HDQ >= 16 ? HDQ : 16;      // columns per flag slot
  constexpr int NHW = NB / NBH;                  // flag slots per wave tile
  bool normed[NHW];
  int nwreg[NHW];                               // 0: q weights, 1: k weights
  float nwv[NB][4];
  if constexpr (HDQ > 0) {
#pragma unroll
    for (int h = 0; h < NHW; ++h) {
      const int c0 = nw0 + h * HSP;
      const int region = c0 / ea.C;  // 0: q, 1: k, 2: v
      normed[h] = region < 2 && c0 < N;
      nwreg[h] = region == 0 ? 0 : 1;
    }
  }

  // this thread's parameter element, loaded here and parked in LDS once the
  // operand ring is free (see the write-out)
  float p_bias = 0.f, p_nw = 0.f, p_rs = 1.f;
  if constexpr (EPI != EPI_NONE && PLDS) {
    const int n = n0 + tid;
    p_bias = tid < BN && n < N ? to_f32(((const T*)ea.bias)[n]) : 0.f;
  }
  if constexpr (HDQ > 0) {
    if (tid < 2 * HDQ) p_nw = to_f32(((const T*)(tid < HDQ ? ea.qn_w : ea.kn_w))[tid % HDQ]);
  }
  if constexpr (PRE == PRE_ROWSCALE) {
    // row m0 + tid's norm from the producer's partial sums of squares, added
    // in a fixed order (rows past M read row 0 and are never stored)
    const int m = m0 + (tid < BM ? tid : 0);
    const float* pp = ea.row_sumsq + (int64_t)(m < M ? m : 0) * ea.nparts;
    float ss = 0.f;
    int q = 0;
    if ((ea.nparts & 3) == 0) {
      for (; q < ea.nparts; q += 4) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(pp + q);
        ss += (v[0] + v[1]) + (v[2] + v[3]);
      }
    }
    for (; q < ea.nparts; ++q) ss += pp[q];
    p_rs = 1.0f / sqrtf(ss / (float)K + ea.eps);
  }

  // PRE_ROWSCALE: the row scales of this lane's rows (from LDS, below)
  float rsr[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) rsr[mb] = 1.f;
  // 1. epilogue math of row block mb in the fragment layout (bias, row scale,
  // head norm, GELU), evaluated where the block is staged
  auto row_values = [&](int mb, float (&v)[NB][4]) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int r = 0; r < 4; ++r) v[nb][r] = (PRE != PRE_NONE ? acc[nb][mb][r] * rsr[mb] : acc[nb][mb][r]) + bv[nb][r];

    if constexpr (HDQ > 0) {
      // sum of squares of each head: local over its blocks, then across the
      // four lane groups holding the same row (xor 16, xor 32)
      float ss[NHW];
#pragma unroll
      for (int h = 0; h < NHW; ++h) {
        float sh = 0.f;
#pragma unroll
        for (int b = 0; b < NBH; ++b)
#pragma unroll
          for (int r = 0; r < 4; ++r) sh = fmaf(v[h * NBH + b][r], v[h * NBH + b][r], sh);
        if constexpr (HDQ >= 16) ss[h] = rows4_sum(sh);
        else if constexpr (HDQ == 8) ss[h] = rows2_sum(sh);
        else ss[h] = sh;
      }
#pragma unroll
      for (int h = 0; h < NHW; ++h) {
        if (normed[h]) {
          // x * rsqrt(mean(x^2) + eps), then * weight, as RMSNorm
          const float rs = __builtin_amdgcn_rsqf(ss[h] * (1.0f / (float)HDQ) + ea.eps);
#pragma unroll
          for (int b = 0; b < NBH; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) v[h * NBH + b][r] = (v[h * NBH + b][r] * rs) * nwv[h * NBH + b][r];
        }
      }
    }
    if constexpr (EPI == EPI_BIAS_GELU) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int r = 0; r < 4; ++r) v[nb][r] = sizeof(T) == 2 ? gelu_erf_bf16(v[nb][r]) : gelu_erf(v[nb][r]);
    } else if constexpr (EPI == EPI_BIAS_GELU_TANH) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int r = 0; r < 4; ++r) v[nb][r] = gelu_tanh(v[nb][r]);
    }
  };

  // 2. write-out through LDS: the waves owning the staged rows store their
  // values in the fragment layout (output dtype), which frees the
  // accumulators, then every wave copies whole rows out with 16-byte lane
  // accesses (fully coalesced) in batches of BATCH rows, adding the residual
  // there.  A batch's output rows (the window -> token map for the scatter)
  // and residual rows are loaded one batch ahead, the first batch's before
  // the staging writes; the loads use clamped addresses (no branches), only
  // the stores are predicated.
  constexpr int VEC = 16 / sizeof(T);                 // elements per 16-byte chunk
  constexpr int LPR = BN / VEC;                       // lanes per output row
  constexpr int RPI = 64 / LPR;                       // rows per copy instruction (1, 2 or 4)
  constexpr int ITER = S::ROWS / NW / RPI;            // copy instructions per wave per pass
  constexpr int BATCH = 8;                            // rows loaded one batch ahead (at most)
  constexpr bool SCAT = EPI == EPI_SCATTER_RESIDUAL;
  constexpr bool REMAP = EPI == EPI_REMAP_RESIDUAL;
  constexpr bool TOK = EPI == EPI_TOKEN_RESIDUAL;
  constexpr bool TOWIN = EPI == EPI_WINDOW_RESIDUAL;
  constexpr bool RES = EPI == EPI_BIAS_RESIDUAL || SCAT || REMAP || TOK || TOWIN || EPI == EPI_RES_SUMSQ;
  // row sums of squares of the stored rows (optional for the scatter)
  constexpr bool SUMSQ = SCAT || REMAP || TOWIN || EPI == EPI_RES_SUMSQ;
  NSW_WAIT_VMCNT(0);                                  // the copies past the last stage
  NSW_WAIT_LGKMCNT0();
  wg_barrier();                                       // the operand ring is no longer read
  if constexpr (PLDS) {
    // epilogue parameters, one element per thread: the tile's bias values,
    // the q and k norm weights, the row scales
    float* prm = reinterpret_cast<float*>(smem + S::PARAM_LDS);
    if constexpr (EPI != EPI_NONE) {
      if (tid < BN) prm[tid] = p_bias;
    }
    if constexpr (HDQ > 0) {
      if (tid < 2 * HDQ) prm[PRM_NW + tid] = p_nw;
    }
    if constexpr (PRE == PRE_ROWSCALE) {
      if (tid < BM) prm[PRM_RS + tid] = p_rs;
    }
    NSW_WAIT_LGKMCNT0();
    wg_barrier();
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const f32x4 b4 = EPI != EPI_NONE ? *reinterpret_cast<const f32x4*>(prm + wn * WTN + nb * 16 + fg * 4)
                                       : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int r = 0; r < 4; ++r) bv[nb][r] = b4[r];
    }
    if constexpr (HDQ > 0) {
#pragma unroll
      for (int h = 0; h < NHW; ++h)
#pragma unroll
        for (int b = 0; b < NBH; ++b) {
          const int dcol = HDQ >= 16 ? b * 16 + fg * 4 : (fg * 4) % HDQ;   // column within the head
          const f32x4 w4 = *reinterpret_cast<const f32x4*>(prm + PRM_NW + nwreg[h] * HDQ + dcol);
#pragma unroll
          for (int r = 0; r < 4; ++r) nwv[h * NBH + b][r] = w4[r];
        }
    }
    if constexpr (PRE == PRE_ROWSCALE) {
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) rsr[mb] = prm[PRM_RS + wm * WTM + mb * 16 + frow];
    }
  }
  char* stg = smem;
  const int lrow = lane / LPR;                        // row of this lane within an instruction
  const int col = (lane % LPR) * VEC;                 // first tile column of this lane
  const int n = n0 + col;
  const int nc = n < N ? n : 0;                       // clamped column for loads
  // Phases: with the whole tile staged at once (bf16), staging and copy-out
  // run in NPH phases of MB / NPH row blocks per wave row, and a
  // phase's copy-out (LDS reads, global stores in flight) is followed by
  // the staging of the next phase's rows, so that the epilogue math (VALU)
  // overlaps the stores of the rows before it.  Phase p covers the tile
  // rows [p RHP, (p + 1) RHP) of every wave row; its copy-out gives each
  // wave WGM RHP / NW consecutive rows of one of them.
  constexpr int NPH = (S::PASSES == 1 && EPI != EPI_UNPATCH) ? (MB < 4 ? MB : 4) : 1;
  constexpr int IPP = ITER / NPH;                     // copy instructions per wave and phase
  constexpr int BAT = IPP < BATCH ? IPP : BATCH;      // rows loaded one batch ahead
  constexpr int NBP = IPP / BAT;                      // batches per phase
  constexpr int NBT = NPH * NBP;                      // batches per pass
  constexpr int RHP = WTM / NPH;                      // rows of a wave row per phase
  static_assert(ITER % NPH == 0 && IPP % BAT == 0 && (NPH == 1 || NW * IPP * RPI == WGM * RHP), "phases");
#pragma unroll
  for (int pass = 0; pass < S::PASSES; ++pass) {
    const int prow0 = pass * S::ROWS;                 // first tile row of this pass
    // tile row of the j-th row of phase p's copy-out (j = wave IPP RPI + ...)
    auto tile_row = [&](int p, int j) {
      return prow0 + (NPH == 1 ? j : (j / RHP) * WTM + p * RHP + j % RHP);
    };
    int orow[2][BAT];                                 // output row (token for the scatter) per batch row
    u32x4 rres[2][RES ? BAT : 1];
    float ssacc = 0.f;                                // row sums of squares of the pass (SUMSQ)
    // Row maps: the wave copies ITER * RPI (<= 64) rows per pass, so lane l
    // maps the wave's l-th row once and every copy instruction takes its
    // rows' targets from those lanes (v_readlane) instead of all 32 or 64
    // lanes of a row evaluating the same map.
    constexpr bool MAPPED = SCAT || TOK || REMAP || TOWIN;
    constexpr int WROWS = ITER * RPI;                 // rows per wave per pass
    static_assert(RPI <= 2 || (!MAPPED && !SUMSQ), "mapped rows and row sums take 1 or 2 rows per instruction");
    static_assert(!SUMSQ || 32 * VEC <= BN, "a part of the row sums (512 bytes) lies in one tile");
    static_assert(WROWS <= 64, "one row per lane");
    // the wave's l-th row (l < WROWS): phase l / (IPP RPI), j = wave IPP RPI + l % (IPP RPI)
    auto wave_row = [&](int l) { return tile_row(l / (IPP * RPI), wave * IPP * RPI + l % (IPP * RPI)); };
    int lmap = 0;
    if constexpr (MAPPED) {
      int mm = m0 + wave_row(lane % WROWS);
      mm = mm < M ? mm : M - 1;
      if constexpr (REMAP) lmap = (int)ea.geom.row_of_row_shift(mm, ea.dh, ea.dw);
      else if constexpr (TOWIN) lmap = (int)ea.geom.row_of_token(mm);
      else lmap = (int)ea.geom.token_of_row(mm);
    }
    // batch g, row b: phase g / NBP, instruction qq of the phase; its rows
    // are the wave's rows ql and ql + 1 (bf16) in the order of wave_row
    auto prefetch = [&](int g, int slot) {
#pragma unroll
      for (int b = 0; b < BAT; ++b) {
        const int ph = g / NBP, qq = (g % NBP) * BAT + b;
        const int ql = (ph * IPP + qq) * RPI;         // lane of this instruction's first row
        int m = m0 + tile_row(ph, wave * IPP * RPI + qq * RPI + lrow);
        m = m < M ? m : M - 1;
        if constexpr (MAPPED) {
          const int a0 = __builtin_amdgcn_readlane(lmap, ql);
          if constexpr (RPI == 2) {
            const int a1 = __builtin_amdgcn_readlane(lmap, ql + 1);
            orow[slot][b] = lrow ? a1 : a0;
          } else {
            orow[slot][b] = a0;
          }
        } else {
          orow[slot][b] = m;
        }
        // the residual row: the output row for the scatter, row m otherwise
        const int rrow = SCAT ? orow[slot][b] : m;
        if constexpr (RES)
          rres[slot][b] = *reinterpret_cast<const u32x4*>((const T*)ea.residual + (int64_t)rrow * N + nc);
      }
    };
    // epilogue math of phase p's row blocks, stored in the fragment layout
    auto stage = [&](int p) {
#pragma unroll
      for (int mb = p * (MB / NPH); mb < (p + 1) * (MB / NPH); ++mb) {
        const int trow = wm * WTM + mb * 16 + frow - prow0;
        if (wm * WTM + mb * 16 - prow0 >= 0 && wm * WTM + mb * 16 - prow0 < S::ROWS) {   // wave-uniform
          float v[NB][4];
          row_values(mb, v);
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) store4<T>(reinterpret_cast<T*>(stg + trow * S::STRIDE) + wn * WTN + nb * 16 + fg * 4, v[nb]);
        }
      }
    };
    prefetch(0, 0);
    stage(0);
    wg_barrier();
    if (pass == 0) NSW_STAMP(ts[3]);
    if constexpr (EPI == EPI_UNPATCH) {
      switch (ea.img_p) {
        case 1: unpatch_copy_out<T, TC, 1>(stg, ea, M, N, m0 + prow0, n0, tid); break;
        case 2: unpatch_copy_out<T, TC, 2>(stg, ea, M, N, m0 + prow0, n0, tid); break;
        case 4: unpatch_copy_out<T, TC, 4>(stg, ea, M, N, m0 + prow0, n0, tid); break;
        case 8: unpatch_copy_out<T, TC, 8>(stg, ea, M, N, m0 + prow0, n0, tid); break;
        default:
          if constexpr (BN >= 256) unpatch_copy_out<T, TC, 16>(stg, ea, M, N, m0 + prow0, n0, tid);
      }
      if (pass + 1 < S::PASSES) wg_barrier();        // before the next pass overwrites the staging rows
      continue;
    }
#pragma unroll
    for (int g = 0; g < NBT; ++g) {
      const int cur = g & 1;
      if (g + 1 < NBT) prefetch(g + 1, cur ^ 1);
      const int ph = g / NBP;
      u32x4 ov[BAT];
#pragma unroll
      for (int b = 0; b < BAT; ++b) {
        const int rl = tile_row(ph, wave * IPP * RPI + ((g % NBP) * BAT + b) * RPI + lrow) - prow0;
        ov[b] = *reinterpret_cast<const u32x4*>(stg + rl * S::STRIDE + col * (int)sizeof(T));
      }
#pragma unroll
      for (int b = 0; b < BAT; ++b) {
        const int qq = (g % NBP) * BAT + b;
        const int m = m0 + tile_row(ph, wave * IPP * RPI + qq * RPI + lrow);
        const bool ok = m < M && n < N;
        float ssq = 0.f;                              // sum of squares of this lane's stored values
        if constexpr (RES) {
          float o[VEC], rv[VEC];
          if constexpr (sizeof(T) == 2) {
            const bf16x8 ob = __builtin_bit_cast(bf16x8, ov[b]);
            const bf16x8 rb = __builtin_bit_cast(bf16x8, rres[cur][b]);
#pragma unroll
            for (int e = 0; e < VEC; ++e) { o[e] = (float)ob[e]; rv[e] = (float)rb[e]; }
          } else {
            const f32x4 of = __builtin_bit_cast(f32x4, ov[b]);
            const f32x4 rf = __builtin_bit_cast(f32x4, rres[cur][b]);
#pragma unroll
            for (int e = 0; e < VEC; ++e) { o[e] = of[e]; rv[e] = rf[e]; }
          }
#pragma unroll
          for (int e = 0; e < VEC; ++e) o[e] += rv[e];
          if (ok) store16<T>(Y + (int64_t)orow[cur][b] * N + n, o);
          if constexpr (SUMSQ) {
            // only stored elements count (lanes past N or rows past M add 0)
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
              const float r = sizeof(T) == 2 ? (float)(T)o[e] : o[e];   // the stored value
              ssq = fmaf(r, r, ssq);
            }
            if (!ok) ssq = 0.f;
          }
        } else {
          // non-temporal: the tile is not read again by this kernel, and the
          // outputs without a residual (qkv, the MLP hidden rows: 398 / 531
          // MB at config 2) exceed the last-level cache; streaming them past
          // L2 made these GEMMs 4-5% faster (fc1 504 -> 481 us, bit-identical;
          // the residual epilogues, whose 133 MB outputs the next kernel
          // reads, showed no gain and keep ordinary stores)
          if (ok) __builtin_nontemporal_store(ov[b], reinterpret_cast<u32x4*>(Y + (int64_t)orow[cur][b] * N + n));
        }
        if constexpr (SUMSQ) {
          // partial sum of squares over 32 lanes (32 * VEC columns, one float
          // per 512 bytes of output row): the two 16-lane row sums of each
          // half wave, even row first, parked in lane ql + half (bf16: the
          // wave's rows ql, ql + 1; fp32: row ql, half = part) of ssacc,
          // which is stored once per pass
          if (!SCAT || ea.row_sumsq != nullptr) {
            const int ri = __builtin_bit_cast(int, row16_sum(ssq));
            const float sa = __builtin_bit_cast(float, __builtin_amdgcn_readlane(ri, 0)) +
                             __builtin_bit_cast(float, __builtin_amdgcn_readlane(ri, 16));
            const float sb = __builtin_bit_cast(float, __builtin_amdgcn_readlane(ri, 32)) +
                             __builtin_bit_cast(float, __builtin_amdgcn_readlane(ri, 48));
            const int ql = (ph * IPP + qq) * RPI;
            constexpr int HB = RPI == 2 ? 1 : 32;       // lane offset of the upper half's value
            ssacc = lane == ql ? sa : ssacc;
            ssacc = lane == ql + HB ? sb : ssacc;
          }
        }
      }
      // the next phase's rows: their math runs while this phase's stores drain
      if ((g + 1) % NBP == 0 && g + 1 < NBT) {
        stage((g + 1) / NBP);
        wg_barrier();
      }
    }
    if constexpr (SUMSQ) {
      // one store of the pass's row sums per wave: bf16, lane l < WROWS
      // holds the wave's row l (part n0 / 256); fp32, lane l with l % 32 <
      // WROWS holds the wave's row l % 32, part n0 / 128 + l / 32
      if (!SCAT || ea.row_sumsq != nullptr) {
        const int rw = RPI == 2 ? lane : (lane & 31);
        const int m = m0 + wave_row(rw < WROWS ? rw : 0);
        const int pcol = n0 + (RPI == 2 ? 0 : (lane >> 5) * 32 * VEC);   // first column of the part
        const int orw = MAPPED ? lmap : m;                                 // lmap: row lane % WROWS (= rw here)
        if (rw < WROWS && m < M && pcol < N) ea.row_sumsq[(int64_t)orw * ea.nparts + pcol / (32 * VEC)] = ssacc;
      }
    }
    if (pass + 1 < S::PASSES) wg_barrier();          // before the next pass overwrites the staging rows
  }
#if NSW_GEMM_STAMPS
  NSW_STAMP(ts[4]);
  if (tid == 0 && tile < NSW_STAMP_TILES) {
    uint64_t* o = nsw_gemm_stamps + (size_t)tile * 8;
#pragma unroll
    for (int i = 0; i < 5; ++i) o[i] = ts[i];
    o[5] = (uint64_t)__builtin_amdgcn_s_getreg((31 << 11) | 4);    // HW_ID
    o[6] = (uint64_t)__builtin_amdgcn_s_getreg((31 << 11) | 20);   // XCC_ID
    o[7] = blockIdx.x;
  }
#endif
}

template <typename T, int EPI, int PRE, class TC>
int launch_tile(const void* x, const void* w, void* y, int64_t M, int64_t N, int64_t K, const EpiArgs& ea,
                       hipStream_t st, const char* what) {
  const int64_t tiles = ((M + TC::BM - 1) / TC::BM) * ((N + TC::BN - 1) / TC::BN);
  NSW_CHECK_ARG(tiles < (1LL << 31), "%s: too many tiles", what);
  hipLaunchKernelGGL((gemm_kernel<T, EPI, PRE, TC>), dim3((unsigned)tiles), dim3(TC::NW * 64), 0, st, (const T*)x,
                     (const T*)w, (T*)y, (int)M, (int)N, (int)K, ea);
  return check_launch(what);
}

}  // namespace nsw

#define NSW_GEMM_INSTANCE(EPI, PRE)                                                                          \
  template int launch_tile<NSW_GEMM_T, EPI, PRE, TileChoice<NSW_GEMM_T, EPI>::NSW_GEMM_SIZE>(                \
      const void*, const void*, void*, int64_t, int64_t, int64_t, const EpiArgs&, hipStream_t, const char*);
