// Fused-part path: dense 2^k x 2^k unitary applied on the gfx950 matrix cores.
//
// The state viewed through a part with qubit set Q (k = |Q|) is a batch of
// 2^(n-k) vectors of length D = 2^k; the fused unitary U maps each of them, so
// the pass is the complex GEMM  Y = U X  with X = D x 2^(n-k). A workgroup
// owns a D x C tile of X whose C columns run along the lowest slots outside Q
// (contiguous in HBM), stages it in LDS, and each of its D/16 waves computes
// 16 rows of Y with 16x16x4 MFMAs, its slice of U held in registers for the
// whole (persistent) launch.
//
// MFMA 16x16x4 operand layouts (checked on gfx950 with a lane probe): lane l
// holds A[l%16][l/16] and B[l/16][l%16]; result item i of lane l is
// D[4*(l/16) + i][l%16] for the f32 instruction but D[l/16 + 4*i][l%16] for
// the f64 one.
//
//  * HSV_FUSED_F64: v_mfma_f64_16x16x4_f64, FP64 products and accumulation;
//    most parts as 4-qubit steps on a tile (k_fused_tile, below).
//  * HSV_FUSED_F32SPLIT: the same FP64 steps where they are the faster way
//    (15 parts of 6 qubits at 25 qubits, read-outs included, 9.6 -> 4.3 ms; 3.0
//    since zero tiles are skipped), and the more exact one; other parts v_mfma_f32_16x16x4_f32 on hi/lo FP32 splits of U and
//    X (x = hi + lo, hi = fp32(x), lo = fp32(x - hi)); each real product is
//    hi*hi + hi*lo + lo*hi, accumulated in FP32; the result is stored back in
//    the state's precision.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#include "../../include/hsv.h"
#include "fused.hpp"
#include "kernels.hpp"
#include "partition.hpp"

namespace hsv {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

struct FusedArgs {
  uint64_t ntiles;
  uint64_t outer_mask;
  int C;       // tile columns = 16 * NC
  int logC;
  int NC;
};

constexpr int kFusedMaxC = 128;

template <typename R, int K, bool SPLIT>
__global__ __launch_bounds__(4 * (1 << K)) void k_fused(typename VecT<R>::type* __restrict__ a,
                                                        const double2* __restrict__ U,
                                                        const uint64_t* __restrict__ qoff,
                                                        const uint64_t* __restrict__ toff, FusedArgs f) {
  constexpr int D = 1 << K;
  constexpr int NT = 4 * D;  // D/16 waves of 64 lanes
  constexpr int KS = D / 4;  // k-steps of the 16x16x4 MFMA
  using V = typename VecT<R>::type;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  double2* X = reinterpret_cast<double2*>(smem_raw);  // D x C tile, row-major
  __shared__ uint64_t sq[D];
  __shared__ uint64_t st[kFusedMaxC];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int C = f.C;
  for (int i = threadIdx.x; i < D; i += NT) sq[i] = qoff[i];
  for (int i = threadIdx.x; i < C; i += NT) st[i] = toff[i];

  // A-operand fragments: lane holds U[16*wave + lane%16][4*ks + lane/16].
  const int arow = 16 * wave + (lane & 15);
  const int akk = lane >> 4;
  double ar[SPLIT ? 1 : KS], ai[SPLIT ? 1 : KS];
  float arh[SPLIT ? KS : 1], arl[SPLIT ? KS : 1], aih[SPLIT ? KS : 1], ail[SPLIT ? KS : 1];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const double2 u = U[arow * D + 4 * ks + akk];
    if constexpr (SPLIT) {
      arh[ks] = (float)u.x; arl[ks] = (float)(u.x - (double)arh[ks]);
      aih[ks] = (float)u.y; ail[ks] = (float)(u.y - (double)aih[ks]);
    } else {
      ar[ks] = u.x; ai[ks] = u.y;
    }
  }
  const int ccol = lane & 15;  // B column / D column within a 16-wide block
  const int krow = lane >> 4;  // B row within a k-step; D row group
  for (uint64_t t = blockIdx.x; t < f.ntiles; t += gridDim.x) {
    const uint64_t base = pdep64(t, f.outer_mask);
    __syncthreads();  // the previous tile's LDS reads are done
    for (int e = threadIdx.x; e < D * C; e += NT) {
      const int r = e >> f.logC, c = e & (C - 1);
      const V v = a[base + sq[r] + st[c]];
      X[e] = make_double2((double)v.x, (double)v.y);
    }
    __syncthreads();
    for (int cb = 0; cb < f.NC; ++cb) {
      if constexpr (SPLIT) {
        v4f accR = {0, 0, 0, 0}, accT = {0, 0, 0, 0}, accI = {0, 0, 0, 0};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const double2 x = X[(4 * ks + krow) * C + 16 * cb + ccol];
          const float xrh = (float)x.x, xrl = (float)(x.x - (double)xrh);
          const float xih = (float)x.y, xil = (float)(x.y - (double)xih);
          // Re: Ur*Xr - Ui*Xi ; Im: Ur*Xi + Ui*Xr (three split products each)
          accR = __builtin_amdgcn_mfma_f32_16x16x4f32(arh[ks], xrh, accR, 0, 0, 0);
          accR = __builtin_amdgcn_mfma_f32_16x16x4f32(arh[ks], xrl, accR, 0, 0, 0);
          accR = __builtin_amdgcn_mfma_f32_16x16x4f32(arl[ks], xrh, accR, 0, 0, 0);
          accT = __builtin_amdgcn_mfma_f32_16x16x4f32(aih[ks], xih, accT, 0, 0, 0);
          accT = __builtin_amdgcn_mfma_f32_16x16x4f32(aih[ks], xil, accT, 0, 0, 0);
          accT = __builtin_amdgcn_mfma_f32_16x16x4f32(ail[ks], xih, accT, 0, 0, 0);
          accI = __builtin_amdgcn_mfma_f32_16x16x4f32(arh[ks], xih, accI, 0, 0, 0);
          accI = __builtin_amdgcn_mfma_f32_16x16x4f32(arh[ks], xil, accI, 0, 0, 0);
          accI = __builtin_amdgcn_mfma_f32_16x16x4f32(arl[ks], xih, accI, 0, 0, 0);
          accI = __builtin_amdgcn_mfma_f32_16x16x4f32(aih[ks], xrh, accI, 0, 0, 0);
          accI = __builtin_amdgcn_mfma_f32_16x16x4f32(aih[ks], xrl, accI, 0, 0, 0);
          accI = __builtin_amdgcn_mfma_f32_16x16x4f32(ail[ks], xrh, accI, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int row = 16 * wave + 4 * krow + i;
          const int col = 16 * cb + ccol;
          V o;
          o.x = (R)((double)accR[i] - (double)accT[i]);
          o.y = (R)accI[i];
          a[base + sq[row] + st[col]] = o;
        }
      } else {
        v4d accR = {0, 0, 0, 0}, accT = {0, 0, 0, 0}, accI = {0, 0, 0, 0};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const double2 x = X[(4 * ks + krow) * C + 16 * cb + ccol];
          accR = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[ks], x.x, accR, 0, 0, 0);
          accT = __builtin_amdgcn_mfma_f64_16x16x4f64(ai[ks], x.y, accT, 0, 0, 0);
          accI = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[ks], x.y, accI, 0, 0, 0);
          accI = __builtin_amdgcn_mfma_f64_16x16x4f64(ai[ks], x.x, accI, 0, 0, 0);
        }
        // f64 result layout differs from f32: item i of lane l is row l/16 + 4i
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int row = 16 * wave + krow + 4 * i;
          const int col = 16 * cb + ccol;
          V o;
          o.x = (R)(accR[i] - accT[i]);
          o.y = (R)accI[i];
          a[base + sq[row] + st[col]] = o;
        }
      }
    }
  }
}

// ---- FP64 fused path, steps on a tile ------------------------------------------
// A part of up to 7 qubits as one dense 2^K x 2^K product costs 8 * 2^K flops
// an amplitude, most of them on the zeros of gates that touch few of its
// qubits. Here the host cuts the part into steps of at most 4 qubits (the
// grouping of the wide BF16-split parts), each a 16 x 16 unitary: 128 flops an
// amplitude and step, one v_mfma_f64_16x16x4_f64 row block, no padding. A
// workgroup owns a tile of 4096 amplitudes (the part's qubits and the lowest
// other slots, so 512-byte runs in complex128) in LDS as FP64, applies the
// steps there in place, a barrier between them, and stores the tile: one pass
// over the state as before. 64 KB of LDS: two workgroups per CU, one computing
// while the other loads or stores. Per tile and CU the pass has 5.3 us of HBM
// time and 1.7 us of matrix time per step, so it is bound by HBM up to about
// three steps. Measured at 28 qubits complex128: 7-qubit QFT
// parts of 2 to 5 steps 2.23 ms on average (3.8 TB/s) against 5.68 ms for the
// dense product (48 TFLOP/s of FP64 MFMA); the state's error against extended
// precision is the dense product's or less (4.4e-16 / 4.7e-16 over a 14-qubit
// QFT, 8.7e-16 / 1.07e-15 over 8 layers).
//
// Step row r sits at tile offset rt[r], column c = 16 cb + l at cth[cb] ^
// ctl[l], all already swizzled (tile_sw is linear). Lane l holds rows l/16 +
// 4 i of column l%16 as operand (k = 4 ks + l/16) and as result, so a wave
// updates its columns in place.
struct TileStep {
  uint16_t rt[16], ctl[16], cth[16];
};
struct TileAddr {
  uint64_t alo[64], ahi[64];  // address offset of tile index bits 0-5 / 6-11
};
constexpr int kTileStepsMax = 8;
constexpr int kTileThreads = 512;

template <typename R>
__global__ __launch_bounds__(kTileThreads) __attribute__((amdgpu_waves_per_eu(4))) void k_fused_tile(
    typename VecT<R>::type* __restrict__ a, const TileAddr* __restrict__ addr, const TileStep* __restrict__ steps,
    const double2* __restrict__ ufrag, int nsteps, uint64_t outer_mask, uint64_t top) {
  using V = typename VecT<R>::type;
  constexpr int PER = 4096 / kTileThreads, W = kTileThreads / 64, CBW = 16 / W;
  __shared__ double2 ys[4096];
  __shared__ TileAddr ad;
  __shared__ TileStep st[kTileStepsMax];
  {
    const uint32_t* src = reinterpret_cast<const uint32_t*>(addr);
    uint32_t* dst = reinterpret_cast<uint32_t*>(&ad);
    for (int i = threadIdx.x; i < (int)(sizeof(TileAddr) / 4); i += kTileThreads) dst[i] = src[i];
    src = reinterpret_cast<const uint32_t*>(steps);
    dst = reinterpret_cast<uint32_t*>(st);
    for (int i = threadIdx.x; i < nsteps * (int)(sizeof(TileStep) / 4); i += kTileThreads) dst[i] = src[i];
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, cc = lane & 15;
  const uint64_t base = tile_base(blockIdx.x, outer_mask, top) + ad.alo[lane];
  {
    V raw[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) raw[j] = ld_stream<R>(&a[base + ad.ahi[wave + W * j]]);
#pragma unroll
    for (int j = 0; j < PER; ++j)
      ys[tile_sw(threadIdx.x + kTileThreads * j)] = make_double2((double)raw[j].x, (double)raw[j].y);
  }
  for (int s = 0; s < nsteps; ++s) {
    double2 u[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) u[ks] = ufrag[(s * 4 + ks) * 64 + lane];  // in flight over the barrier
    __syncthreads();  // the tile, or the previous step's results, is in LDS
    const TileStep& S = st[s];
    uint32_t row[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) row[i] = S.rt[4 * i + g] ^ S.ctl[cc];
#pragma unroll
    for (int w = 0; w < CBW; ++w) {
      const uint32_t cb = S.cth[wave * CBW + w];
      double2 x[4];
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) x[ks] = ys[row[ks] ^ cb];
      v4d accR = {0, 0, 0, 0}, accT = {0, 0, 0, 0}, accI = {0, 0, 0, 0}, accJ = {0, 0, 0, 0};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        accR = __builtin_amdgcn_mfma_f64_16x16x4f64(u[ks].x, x[ks].x, accR, 0, 0, 0);
        accT = __builtin_amdgcn_mfma_f64_16x16x4f64(u[ks].y, x[ks].y, accT, 0, 0, 0);
        accI = __builtin_amdgcn_mfma_f64_16x16x4f64(u[ks].x, x[ks].y, accI, 0, 0, 0);
        accJ = __builtin_amdgcn_mfma_f64_16x16x4f64(u[ks].y, x[ks].x, accJ, 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) ys[row[i] ^ cb] = make_double2(accR[i] - accT[i], accI[i] + accJ[i]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const double2 y = ys[tile_sw(threadIdx.x + kTileThreads * j)];
    V o;
    o.x = (R)y.x;
    o.y = (R)y.y;
    st_stream<R>(&a[base + ad.ahi[wave + W * j]], o);
  }
}

// ---- BF16-split fused path ------------------------------------------------------
// gfx950's dense BF16 rate is 16x its FP32 rate, so here U and X are split
// into BF16 pairs (v = hi + lo, hi = bf16(v), lo = bf16(v - hi): 16
// significant bits) and every real product is hi*hi + hi*lo + lo*hi on
// v_mfma_f32_16x16x32_bf16, accumulated in FP32. U's fragments live in LDS
// for the whole (persistent) launch; each wave owns column blocks of 16
// columns (16 amplitudes along the lowest slots outside the part) and
// streams their D rows from HBM straight into B operands, 32 rows per
// k-step, the next k-step's loads in flight while the current one runs.
//
// 16x16x32 operand layouts (checked on gfx950 with a lane probe): lane l holds
// A[l%16][8*(l/16) + e] and B[8*(l/16) + e][l%16] for e = 0..7 (any k order
// shared by A and B gives the same product), and result item i of lane l is
// D[4*(l/16) + i][l%16].
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf2v __attribute__((ext_vector_type(2)));
typedef float f2v __attribute__((ext_vector_type(2)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));

// Two floats to their BF16 hi parts (round to nearest even, packed in one
// dword as element pair 2j, 2j+1 of a bf8 operand) and the BF16 of the
// remainders: a = hi_a + lo_a to 16 significant bits. One v_cvt_pk_bf16_f32
// per pair for each of hi and lo; hi back to FP32 is a shift or a mask.
__device__ __forceinline__ void split_pair(float a, float b, uint32_t* hi, uint32_t* lo) {
  const f2v ab = {a, b};
  const uint32_t h = __builtin_bit_cast(uint32_t, __builtin_convertvector(ab, bf2v));
  const f2v rest = {a - __builtin_bit_cast(float, h << 16), b - __builtin_bit_cast(float, h & 0xffff0000u)};
  *hi = h;
  *lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(rest, bf2v));
}

// The three-piece split (Henry, Tang and Heinecke, "Leveraging the bfloat16
// artificial intelligence datatype for higher-precision computations",
// ARITH 2019): a = hi + mid + lo with each piece the BF16 of what the
// previous ones leave (both remainders are exact in FP32), 24 significant
// bits in all; the residual is below 2^-26 |a|.
__device__ __forceinline__ void split_pair3(float a, float b, uint32_t* hi, uint32_t* mid, uint32_t* lo) {
  const f2v ab = {a, b};
  const uint32_t h = __builtin_bit_cast(uint32_t, __builtin_convertvector(ab, bf2v));
  const f2v r1 = {a - __builtin_bit_cast(float, h << 16), b - __builtin_bit_cast(float, h & 0xffff0000u)};
  const uint32_t m = __builtin_bit_cast(uint32_t, __builtin_convertvector(r1, bf2v));
  const f2v r2 = {r1[0] - __builtin_bit_cast(float, m << 16), r1[1] - __builtin_bit_cast(float, m & 0xffff0000u)};
  *hi = h;
  *mid = m;
  *lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(r2, bf2v));
}

// 8 complex values (rows of a B operand) to the four BF16 operands: real hi,
// real lo, imaginary hi, imaginary lo.
__device__ __forceinline__ void split_bf8(const float2 (&v)[8], bf8* rh, bf8* rl, bf8* ih, bf8* il) {
  u4v a, b, c, d;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    uint32_t x0, x1, y0, y1;
    split_pair(v[2 * j].x, v[2 * j + 1].x, &x0, &x1);
    split_pair(v[2 * j].y, v[2 * j + 1].y, &y0, &y1);
    a[j] = x0;
    b[j] = x1;
    c[j] = y0;
    d[j] = y1;
  }
  *rh = __builtin_bit_cast(bf8, a);
  *rl = __builtin_bit_cast(bf8, b);
  *ih = __builtin_bit_cast(bf8, c);
  *il = __builtin_bit_cast(bf8, d);
}

// The same with three pieces: real hi, mid, lo, imaginary hi, mid, lo.
__device__ __forceinline__ void split_bf8_3(const float2 (&v)[8], bf8* rh, bf8* rm, bf8* rl, bf8* ih, bf8* im,
                                            bf8* il) {
  u4v a, b, c, d, e, f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    uint32_t x0, x1, x2, y0, y1, y2;
    split_pair3(v[2 * j].x, v[2 * j + 1].x, &x0, &x1, &x2);
    split_pair3(v[2 * j].y, v[2 * j + 1].y, &y0, &y1, &y2);
    a[j] = x0;
    b[j] = x1;
    c[j] = x2;
    d[j] = y0;
    e[j] = y1;
    f[j] = y2;
  }
  *rh = __builtin_bit_cast(bf8, a);
  *rm = __builtin_bit_cast(bf8, b);
  *rl = __builtin_bit_cast(bf8, c);
  *ih = __builtin_bit_cast(bf8, d);
  *im = __builtin_bit_cast(bf8, e);
  *il = __builtin_bit_cast(bf8, f);
}

// Column signs of the three-piece split. column_hash: murmur3's 32-bit
// finaliser of (tile << 8 | column) (columns < 256), once per tile;
// column_sign: 0 or the FP32 sign bit for one step, the top bit of
// (hash ^ step * 0x85EBCA77) * 0x9E3779B1.
__device__ __forceinline__ uint32_t column_hash(uint64_t tile, int col) {
  uint32_t k = uint32_t(tile) << 8 | uint32_t(col);
  k ^= k >> 16;
  k *= 0x85EBCA6Bu;
  k ^= k >> 13;
  k *= 0xC2B2AE35u;
  k ^= k >> 16;
  return k;
}
__device__ __forceinline__ uint32_t column_sign(uint32_t hash, int step) {
  return ((hash ^ (uint32_t(step) * 0x85EBCA77u)) * 0x9E3779B1u) & 0x80000000u;
}

struct BfArgs {
  uint64_t nblocks;     // column blocks of 16 columns
  uint64_t outer_mask;  // outer bits above the 4 column bits
};

constexpr int kBfThreads = 512;

// SWZ: row order of the B operands and of the results. false: lane l, element
// e reads row 8*(l/16) + e of its k-step and stores result item i to row
// 4*(l/16) + i. true: rows (l/16) + 4*e and 4*i + (l/16), so the 4 lanes of
// a column cover 4 consecutive rows in each load and store instruction; the
// host permutes U's columns and rows to match (any k order shared by A and
// B, and any row order of A, leave the product the same up to that order).
template <typename R, int K, bool SWZ>
__global__ __launch_bounds__(kBfThreads) void k_fused_bf(typename VecT<R>::type* __restrict__ a,
                                                       const bf8* __restrict__ ufrag,
                                                       const uint64_t* __restrict__ qoff,
                                                       const uint64_t* __restrict__ toff, BfArgs f) {
  constexpr int D = 1 << K;
  constexpr int RB = D / 16;  // row blocks of the 16x16 result
  constexpr int KS = D / 32;  // k-steps of 32
  using V = typename VecT<R>::type;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  bf8* su = reinterpret_cast<bf8*>(smem_raw);  // [rb][ks][set][lane], set = Ur_h, Ur_l, Ui_h, Ui_l
  __shared__ uint64_t sq[D];
  for (int i = threadIdx.x; i < RB * KS * 4 * 64; i += kBfThreads) su[i] = ufrag[i];
  for (int i = threadIdx.x; i < D; i += kBfThreads) sq[i] = qoff[i];
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int kgrp = lane >> 4;
  const uint64_t coff = toff[lane & 15];
  const uint64_t nw = uint64_t(gridDim.x) * (kBfThreads / 64);
  typedef float v4f_t __attribute__((ext_vector_type(4)));
  // raw: this lane's 8 amplitudes of each k-step (rows 32 ks + 8 kgrp + e,
  // column lane % 16); the next block's are loaded while this one's MFMAs run
  V raw[KS][8];
  uint64_t cb = uint64_t(blockIdx.x) * (kBfThreads / 64) + wave;
  if (cb < f.nblocks) {
    const uint64_t base = pdep64(cb, f.outer_mask) + coff;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int e = 0; e < 8; ++e) raw[ks][e] = a[base + sq[32 * ks + (SWZ ? kgrp + 4 * e : 8 * kgrp + e)]];
  }
  for (; cb < f.nblocks; cb += nw) {
    const uint64_t base = pdep64(cb, f.outer_mask) + coff;
    bf8 xrh[KS], xrl[KS], xih[KS], xil[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float xr = (float)raw[ks][e].x, xi = (float)raw[ks][e].y;
        const __bf16 hr = (__bf16)xr, hi = (__bf16)xi;
        xrh[ks][e] = hr;
        xrl[ks][e] = (__bf16)(xr - (float)hr);
        xih[ks][e] = hi;
        xil[ks][e] = (__bf16)(xi - (float)hi);
      }
    const uint64_t cn = cb + nw;
    if (cn < f.nblocks) {
      const uint64_t nbase = pdep64(cn, f.outer_mask) + coff;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int e = 0; e < 8; ++e) raw[ks][e] = a[nbase + sq[32 * ks + (SWZ ? kgrp + 4 * e : 8 * kgrp + e)]];
    }
    // every row of this column block is in registers now: results can be
    // written as each row block finishes
#pragma unroll 1
    for (int rb = 0; rb < RB; ++rb) {
      v4f_t accR = {0, 0, 0, 0}, accT = {0, 0, 0, 0}, accI = {0, 0, 0, 0};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const bf8* A = su + ((rb * KS + ks) * 4) * 64 + lane;
        const bf8 urh = A[0], url = A[64], uih = A[128], uil = A[192];
        // Re = Ur Xr - Ui Xi ; Im = Ur Xi + Ui Xr, three split products each
        accR = __builtin_amdgcn_mfma_f32_16x16x32_bf16(urh, xrh[ks], accR, 0, 0, 0);
        accR = __builtin_amdgcn_mfma_f32_16x16x32_bf16(urh, xrl[ks], accR, 0, 0, 0);
        accR = __builtin_amdgcn_mfma_f32_16x16x32_bf16(url, xrh[ks], accR, 0, 0, 0);
        accT = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uih, xih[ks], accT, 0, 0, 0);
        accT = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uih, xil[ks], accT, 0, 0, 0);
        accT = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uil, xih[ks], accT, 0, 0, 0);
        accI = __builtin_amdgcn_mfma_f32_16x16x32_bf16(urh, xih[ks], accI, 0, 0, 0);
        accI = __builtin_amdgcn_mfma_f32_16x16x32_bf16(urh, xil[ks], accI, 0, 0, 0);
        accI = __builtin_amdgcn_mfma_f32_16x16x32_bf16(url, xih[ks], accI, 0, 0, 0);
        accI = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uih, xrh[ks], accI, 0, 0, 0);
        accI = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uih, xrl[ks], accI, 0, 0, 0);
        accI = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uil, xrh[ks], accI, 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        V o;
        o.x = (R)(accR[i] - accT[i]);
        o.y = (R)accI[i];
        a[base + sq[16 * rb + (SWZ ? 4 * i + kgrp : 4 * kgrp + i)]] = o;
      }
    }
  }
}

// ---- BF16-split fused path, U-stationary tile form ---------------------------------
// A workgroup (8 waves) owns a tile of 4096 amplitudes: the part's D rows by
// C = 4096 / D columns along the lowest slots outside the part. Tile element
// t (12 bits) maps to the tile's 12 slots in ascending order, so consecutive
// threads load and store consecutive amplitudes. Loaded values are split to
// BF16 and scattered into B-operand fragments in LDS; wave w keeps row block
// w % RB of U in registers (its A fragments) and computes that row block for
// its share of the columns; results go through an FP32 staging tile in LDS
// and are stored back coalesced. LDS: 32 KB of fragments + 32 KB of staging.
struct BfTileTables {
  uint64_t alo[64], ahi[64];    // address offset of tile index bits 0-5 / 6-11
  uint16_t rlo[64], rhi[64];    // row index contribution of those bits
  uint16_t clo[64], chi[64];    // column index contribution
  uint16_t tr[128], tc[128];    // tile index of row r / column c (OR-ed)
};

constexpr int kBfTileThreads = 512;

template <typename R, int K>
__global__ __launch_bounds__(kBfTileThreads) void k_fused_bft(typename VecT<R>::type* __restrict__ a,
                                                            const bf8* __restrict__ ufrag,
                                                            const BfTileTables* __restrict__ tabs,
                                                            uint64_t ntiles, uint64_t outer_mask, uint64_t top,
                                                            int tiles_per_wg) {
  constexpr int D = 1 << K;
  constexpr int RB = D / 16, KS = D / 32;
  constexpr int C = 4096 / D, NCB = C / 16;
  constexpr int W = kBfTileThreads / 64;
  constexpr int CG = W / RB;        // waves sharing one row block
  constexpr int CBW = NCB / CG;     // column blocks per wave
  constexpr int PER = 4096 / kBfTileThreads;
  using V = typename VecT<R>::type;
  __shared__ bf8 xs[KS * NCB * 4 * 64];   // [ks][cb][set][lane], set = Xr_h, Xr_l, Xi_h, Xi_l
  __shared__ float2 ys[4096];             // results in tile order
  __shared__ BfTileTables tb;
  {
    const uint32_t* src = reinterpret_cast<const uint32_t*>(tabs);
    uint32_t* dst = reinterpret_cast<uint32_t*>(&tb);
    for (int i = threadIdx.x; i < (int)(sizeof(BfTileTables) / 4); i += kBfTileThreads) dst[i] = src[i];
  }
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int rb = wave % RB, cg = wave / RB;
  bf8 A[KS][4];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
#pragma unroll
    for (int s = 0; s < 4; ++s) A[ks][s] = ufrag[((rb * KS + ks) * 4 + s) * 64 + lane];
  __syncthreads();
  __bf16* xb = reinterpret_cast<__bf16*>(xs);
  typedef float v4f_t __attribute__((ext_vector_type(4)));
  // consecutive tiles per workgroup, no prefetch (the other workgroups on
  // the CU overlap this one's compute); the U fragments above are loaded
  // once per workgroup
  for (int it = 0; it < tiles_per_wg; ++it) {
    const uint64_t tile = uint64_t(blockIdx.x) * tiles_per_wg + it;
    if (tile >= ntiles) break;  // uniform across the workgroup
    const uint64_t base = tile_base(tile, outer_mask, top);
    V raw[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int t = threadIdx.x + kBfTileThreads * j;
      raw[j] = ld_stream<R>(&a[base + tb.alo[t & 63] + tb.ahi[t >> 6]]);
    }
    __syncthreads();  // the previous tile's stores have read ys (and the xs reads are done)
    // split and scatter this thread's elements into the B fragments:
    // row r = 32 ks + g + 4 e goes to lane 16 g + (c % 16), element e
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int t = threadIdx.x + kBfTileThreads * j;
      const int r = tb.rlo[t & 63] + tb.rhi[t >> 6];
      const int c = tb.clo[t & 63] + tb.chi[t >> 6];
      const int ks = r >> 5, g = r & 3, e = (r >> 2) & 7;
      const int frag = (ks * NCB + (c >> 4)) * 4 * 64 + 16 * g + (c & 15);
      const float xr = (float)raw[j].x, xi = (float)raw[j].y;
      const __bf16 hr = (__bf16)xr, hi = (__bf16)xi;
      xb[(frag + 0 * 64) * 8 + e] = hr;
      xb[(frag + 1 * 64) * 8 + e] = (__bf16)(xr - (float)hr);
      xb[(frag + 2 * 64) * 8 + e] = hi;
      xb[(frag + 3 * 64) * 8 + e] = (__bf16)(xi - (float)hi);
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < CBW; ++w) {
      const int cb = cg * CBW + w;
      v4f_t accR = {0, 0, 0, 0}, accT = {0, 0, 0, 0}, accI = {0, 0, 0, 0};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const bf8* B = xs + (ks * NCB + cb) * 4 * 64 + lane;
        const bf8 xrh = B[0], xrl = B[64], xih = B[128], xil = B[192];
        accR = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[ks][0], xrh, accR, 0, 0, 0);
        accR = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[ks][0], xrl, accR, 0, 0, 0);
        accR = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[ks][1], xrh, accR, 0, 0, 0);
        accT = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[ks][2], xih, accT, 0, 0, 0);
        accT = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[ks][2], xil, accT, 0, 0, 0);
        accT = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[ks][3], xih, accT, 0, 0, 0);
        accI = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[ks][0], xih, accI, 0, 0, 0);
        accI = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[ks][0], xil, accI, 0, 0, 0);
        accI = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[ks][1], xih, accI, 0, 0, 0);
        accI = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[ks][2], xrh, accI, 0, 0, 0);
        accI = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[ks][2], xrl, accI, 0, 0, 0);
        accI = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[ks][3], xrh, accI, 0, 0, 0);
      }
      // item i of lane l: row 16 rb + 4 i + l/16 (the swizzled A rows), column 16 cb + l % 16
      const int col = 16 * cb + (lane & 15);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 16 * rb + 4 * i + (lane >> 4);
        ys[tb.tr[row] | tb.tc[col]] = make_float2(accR[i] - accT[i], accI[i]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int t = threadIdx.x + kBfTileThreads * j;
      const float2 y = ys[t];
      V o;
      o.x = (R)y.x;
      o.y = (R)y.y;
      st_stream<R>(&a[base + tb.alo[t & 63] + tb.ahi[t >> 6]], o);
    }
  }
}

// ---- BF16-split wide parts: 12- to 14-qubit tiles, 5-qubit fused steps ------------
// For a part of 8..14 qubits the host splits the gates into steps of at most
// 5 qubits (the qubit-set closure method), fuses each step into a 32 x 32
// FP64 unitary and sends its BF16 A fragments. A workgroup owns one tile of
// 2^KT amplitudes (the part's qubits, padded with the lowest free ones, in
// ascending order: tile index bit j <-> the j-th of them): it loads the tile
// coalesced into LDS as FP32, applies the steps there one after another
// (rows = the step's 5 tile bits, columns = the other KT - 5; each wave owns
// column blocks of 16 and updates them in place; a barrier between steps),
// and stores the tile back coalesced. One HBM pass per part, the gate work
// on the matrix cores.
//
// LDS bank swizzle: tile element t lives at ys[t ^ h(t >> 4)], h linear over
// GF(2) (swz[] tabulates it; tile bit 4 feeds only bits 0-3, so the map is
// invertible), chosen on the host per part so that the 16
// lanes of a quarter-wave (16 columns of one row) and the two rows of a
// half-wave fall in distinct banks for every step. Because the map is
// linear, a step's row and column offsets are tabulated already swizzled and
// combined with XOR. Without it, a step on the low tile bits reads its
// columns at a stride of 32+ elements: 16-way bank conflicts.
struct PartBfStep {
  uint16_t rt[32];              // swizzled LDS offset of step row r
  uint16_t ctl[16], cth[32];    // of step column c: ctl[c & 15] ^ cth[c >> 4]
};
struct PartBfTables {
  uint64_t alo[64], ahi[256];   // address offset of tile index bits 0-5 / 6-13
  // A layout change moves qubits between the tile's slots: the element
  // stored at tile position u is the one loaded at position plo[u & 63] |
  // phi[u >> 6] (the identity without a change), so the stores stay as
  // coalesced as the loads.
  uint16_t plo[64], phi[256];
  uint8_t swz[1024];            // h(t >> 4): XOR into the low 5 bits of t
};
// 512 threads: 8 amplitudes per thread for 12-qubit tiles, 16 for 13; 1024
// threads (16 amplitudes each) for 14. 12-qubit tiles keep every step's U
// fragments in LDS; 13-qubit tiles (64 KB of FP32 in LDS) either stream them
// (STREAM_U) through one 8 KB buffer, each of 512 threads holding its
// 16-byte share of the next step in a register, so two workgroups fit a CU
// and one computes while the other loads or stores; or keep them resident
// with 1024 threads (8 amplitudes each) and one workgroup per CU, which
// then loads the next tile into registers during the steps, as 12-qubit
// tiles do. A 14-qubit tile (128 KB) fills the CU alone and streams, so its
// compute does not overlap its I/O (66 ms against 54 ms per pass at 33
// qubits): it saves passes only where parts get much wider.
constexpr int part_bf_threads(int kt, bool stream_u) { return kt >= 14 || (kt == 13 && !stream_u) ? 1024 : 512; }
constexpr int kPartBfMaxSteps = 12;
// steps per launch: 8 for the streamed three-piece 13-qubit form (its 12 KB
// fragment buffer leaves room for 8 step tables, two workgroups per CU)
constexpr int part_bf_max_steps(int kt, int np) { return np == 3 && kt == 13 ? 8 : kPartBfMaxSteps; }

// NP: BF16 pieces per value, 2 (hi*hi + hi*lo + lo*hi, 16 significant bits)
// or 3 (the three-piece split: hi*hi, hi*mid, mid*hi, mid*mid, hi*lo, lo*hi,
// 24 bits, FP32-class products; 12-qubit tiles with resident fragments, or
// 13-qubit tiles streaming 12 KB of fragments per step, with at most 8 steps
// per launch so that two workgroups still fit a CU).
template <typename R, int KT, bool STREAM_U, bool U_DIRECT = false, int NP = 2>
// 16 waves per CU (two workgroups of 8, or one of 16): at most 128 VGPRs
__global__ __launch_bounds__(part_bf_threads(KT, STREAM_U)) __attribute__((amdgpu_waves_per_eu(4))) void k_part_bf(typename VecT<R>::type* __restrict__ a,
                                                          const PartBfTables* __restrict__ tabs,
                                                          const PartBfStep* __restrict__ steps_g,
                                                          const bf8* __restrict__ ufrag, int nsteps,
                                                          uint64_t ntiles, uint64_t outer_mask, uint64_t top,
                                                          int tiles_per_wg) {
  constexpr int T = 1 << KT;
  constexpr int NCB = (1 << (KT - 5)) / 16;   // column blocks of a step
  constexpr int NTH = part_bf_threads(KT, STREAM_U);
  constexpr int W = NTH / 64;
  constexpr int CBW = NCB / W;                // column blocks per wave
  constexpr int PER = T / NTH;
  static_assert(KT == 13 || STREAM_U == (KT >= 14), "12-qubit tiles keep U resident, 14-qubit tiles stream it");
  constexpr int STEP_FRAGS = 2 * 2 * NP * 64;  // bf8 per step: [rb][set][lane]
  static_assert(NP == 2 || (NP == 3 && ((KT == 12 && !STREAM_U) || (KT == 13 && STREAM_U && !U_DIRECT))),
                "three pieces: 12-qubit tiles with resident fragments or streamed 13-qubit tiles");
  constexpr int FRPT = (STEP_FRAGS + NTH - 1) / NTH;  // streamed fragments held per thread
  constexpr int MAX_STEPS = part_bf_max_steps(KT, NP);
  static_assert(CBW >= 1 && NCB % W == 0 && PER * NTH == T, "tile shape");
  static_assert(!STREAM_U || STEP_FRAGS <= 2 * NTH, "at most two fragments per thread per step");
  static_assert(!U_DIRECT || STREAM_U, "direct fragment loads replace the streaming buffer");
  constexpr bool SU_BUF = STREAM_U && !U_DIRECT;
  using V = typename VecT<R>::type;
  typedef float v4f_t __attribute__((ext_vector_type(4)));
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ bf8 su_one[SU_BUF ? STEP_FRAGS : 1];
  bf8* su = STREAM_U ? su_one : reinterpret_cast<bf8*>(smem_raw);     // [step][rb][set][lane]
  __shared__ float2 ys[T];
  __shared__ PartBfStep st[MAX_STEPS];
  __shared__ uint64_t alo[64], ahi[T >> 6];
  __shared__ uint16_t plo[64], phi[T >> 6];
  __shared__ uint8_t swz[T >> 4];
  if constexpr (!STREAM_U)
    for (int i = threadIdx.x; i < nsteps * STEP_FRAGS; i += NTH) su[i] = ufrag[i];
  {
    const uint32_t* src = reinterpret_cast<const uint32_t*>(steps_g);
    uint32_t* dst = reinterpret_cast<uint32_t*>(st);
    for (int i = threadIdx.x; i < nsteps * (int)(sizeof(PartBfStep) / 4); i += NTH) dst[i] = src[i];
  }
  for (int i = threadIdx.x; i < 64; i += NTH) alo[i] = tabs->alo[i];
  for (int i = threadIdx.x; i < (T >> 6); i += NTH) ahi[i] = tabs->ahi[i];
  for (int i = threadIdx.x; i < 64; i += NTH) plo[i] = tabs->plo[i];
  for (int i = threadIdx.x; i < (T >> 6); i += NTH) phi[i] = tabs->phi[i];
  for (int i = threadIdx.x; i < (T >> 4); i += NTH) swz[i] = tabs->swz[i];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int g = lane >> 4, cc = lane & 15;
  // A few consecutive tiles per workgroup (tiles_per_wg; the grid covers
  // the rest). With the fragments resident, the next tile's loads are issued
  // before this tile's steps and overlap them. (With streamed fragments the
  // per-step fragment loads would wait behind such a prefetch, so there the
  // other workgroup on the CU provides the overlap.)
  const uint64_t t0 = uint64_t(blockIdx.x) * tiles_per_wg;
  if (t0 >= ntiles) return;  // uniform across the workgroup
  const int nt = (int)min(uint64_t(tiles_per_wg), ntiles - t0);
  bf8 fr[FRPT];  // streamed fragments: this thread's share of the next step
  if constexpr (SU_BUF) {
#pragma unroll
    for (int i = 0; i < FRPT; ++i)
      if (threadIdx.x + NTH * i < STEP_FRAGS) fr[i] = ufrag[threadIdx.x + NTH * i];
  }
  __syncthreads();  // tables ready
  // Thread x handles tile positions t = x + NTH j: t & 63 is its lane and
  // t >> 6 = wave + W j, so the per-j table entries sit at fixed offsets
  // from one base (no per-j address registers).
  const uint64_t a_lo = alo[lane];
  const int p_lo = plo[lane];
  V raw[PER];
  if constexpr (!STREAM_U) {
    const uint64_t base = tile_base(t0, outer_mask, top);
#pragma unroll
    for (int j = 0; j < PER; ++j) raw[j] = ld_stream<R>(&a[base + a_lo + ahi[wave + W * j]]);
  }
  for (int it = 0; it < nt; ++it) {
    const uint64_t base = tile_base(t0 + it, outer_mask, top);
    if constexpr (STREAM_U) {
#pragma unroll
      for (int j = 0; j < PER; ++j) raw[j] = ld_stream<R>(&a[base + a_lo + ahi[wave + W * j]]);
    }
    if (it > 0) __syncthreads();  // the previous tile's stores have read ys
    // t ^ swz[t >> 4] with swz < 32 and NTH j a multiple of 512. The swizzle
    // is linear and t >> 4 = (x >> 4) | (NTH / 16) j with disjoint bits, so
    // swz[t >> 4] = swz[x >> 4] ^ swz[(NTH / 16) j]: one per-thread table
    // read, the rest wave-uniform (scalar loads of the global copy, so no
    // per-j address registers stay live across the tile loop)
    {
      const uint32_t sw_x = swz[threadIdx.x >> 4];
      // swz[(NTH / 16) 2^b], b < log2(PER), read as aligned words
      const uint32_t* sw_words = reinterpret_cast<const uint32_t*>(tabs->swz);
      uint32_t hb[4];
#pragma unroll
      for (int b = 0; b < 4; ++b)
        hb[b] = (1 << b) < PER ? __builtin_amdgcn_readfirstlane(sw_words[((NTH >> 4) << b) >> 2] & 0xffu) : 0u;
#pragma unroll
      for (int j = 0; j < PER; ++j) {
        uint32_t hj = 0;
#pragma unroll
        for (int b = 0; b < 4; ++b)
          if (j >> b & 1) hj ^= hb[b];
        ys[(threadIdx.x ^ sw_x ^ hj) + NTH * j] = make_float2((float)raw[j].x, (float)raw[j].y);
      }
    }
    if (!STREAM_U && it + 1 < nt) {
      const uint64_t nbase = tile_base(t0 + it + 1, outer_mask, top);
#pragma unroll
      for (int j = 0; j < PER; ++j) raw[j] = ld_stream<R>(&a[nbase + a_lo + ahi[wave + W * j]]);
    }
    // three pieces: each of this lane's columns keeps its hash for the tile
    uint32_t colh[NP == 3 ? CBW : 1];
    if constexpr (NP == 3) {
#pragma unroll
      for (int w = 0; w < CBW; ++w) colh[w] = column_hash(t0 + it, 16 * (wave * CBW + w) + cc);
    }
    for (int s = 0; s < nsteps; ++s) {
      const bf8* As;
      bf8 Af[2][4];
      if constexpr (U_DIRECT) {
        // each wave reads the step's fragments straight from L2 into
        // registers, issued before the barrier so that their latency
        // overlaps it
        As = ufrag + s * STEP_FRAGS + lane;
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
#pragma unroll
          for (int q = 0; q < 4; ++q) Af[rb][q] = As[(rb * 4 + q) * 64];
      }
      __syncthreads();  // the tile (or the previous step's results) is in LDS
      const PartBfStep& S = st[s];
      if constexpr (U_DIRECT) {
      } else if constexpr (STREAM_U) {
#pragma unroll
        for (int i = 0; i < FRPT; ++i) {
          const int f = threadIdx.x + NTH * i;
          if (f < STEP_FRAGS) {
            su_one[f] = fr[i];  // every wave is past the previous step's reads
            fr[i] = ufrag[(s + 1 < nsteps ? s + 1 : 0) * STEP_FRAGS + f];
          }
        }
        __syncthreads();
        As = su_one + lane;
      } else {
        As = su + s * STEP_FRAGS + lane;
      }
      // This lane reads rows g + 4e (e = 0..7) of its columns and writes
      // result item i of row block rb to row 16 rb + 4 i + g: the same 8
      // rows, so one set of row offsets serves both. All of the wave's column
      // blocks are read and split before any MFMA and written after them
      // (each wave owns its columns for the whole step), so the blocks'
      // product chains interleave instead of running one block at a time.
      // (two 16-bit offsets per register)
      uint32_t roff2[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) roff2[e] = uint32_t(S.rt[g + 8 * e]) | (uint32_t(S.rt[g + 8 * e + 4]) << 16);
      auto roff = [&](int e) -> uint32_t { return e & 1 ? roff2[e >> 1] >> 16 : roff2[e >> 1] & 0xffffu; };
      uint32_t tc[CBW];
#pragma unroll
      for (int w = 0; w < CBW; ++w) {
        const int col = 16 * (wave * CBW + w) + cc;
        tc[w] = S.ctl[col & 15] ^ S.cth[col >> 4];
      }
      if constexpr (NP == 3) {
        // three pieces: the six products of each real product, smallest
        // first into the FP32 accumulator; one column block at a time (each
        // wave owns its columns, so a block is read, multiplied and written
        // before the next without a hazard), which keeps the eighteen BF16
        // operands of a block and its accumulators within 128 VGPRs.
        // The matrix cores' FP32 accumulation rounds with a small bias of
        // one direction: a pass's error has a component that is the same in
        // every tile and for every input, which later Hadamards (a QFT's)
        // add up onto a few amplitudes. Each column's 32 values are
        // negated before the products and the results negated back, by a
        // sign hashed from (tile, column, step): exact, and bit-identical
        // under unbiased rounding, while the bias of each column then
        // enters with a pseudo-random sign and no longer adds up.
#pragma unroll
        for (int w = 0; w < CBW; ++w) {
          const uint32_t fl = column_sign(colh[w], s);
          bf8 xrh, xrm, xrl, xih, xim, xil;
          {
            float2 v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const float2 y = ys[roff(e) ^ tc[w]];
              v[e] = make_float2(flip_sign(y.x, fl), flip_sign(y.y, fl));
            }
            split_bf8_3(v, &xrh, &xrm, &xrl, &xih, &xim, &xil);
          }
#pragma unroll
          for (int rb = 0; rb < 2; ++rb) {
            const bf8* Ar = As + rb * 6 * 64;
            const bf8 urh = Ar[0], urm = Ar[64], url = Ar[128], uih = Ar[192], uim = Ar[256], uil = Ar[320];
            const v4f_t z = {0, 0, 0, 0};
            v4f_t accR = __builtin_amdgcn_mfma_f32_16x16x32_bf16(urh, xrl, z, 0, 0, 0);
            v4f_t accT = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uih, xil, z, 0, 0, 0);
            v4f_t accI = __builtin_amdgcn_mfma_f32_16x16x32_bf16(urh, xil, z, 0, 0, 0);
            v4f_t accJ = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uih, xrl, z, 0, 0, 0);
            accR = __builtin_amdgcn_mfma_f32_16x16x32_bf16(url, xrh, accR, 0, 0, 0);
            accT = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uil, xih, accT, 0, 0, 0);
            accI = __builtin_amdgcn_mfma_f32_16x16x32_bf16(url, xih, accI, 0, 0, 0);
            accJ = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uil, xrh, accJ, 0, 0, 0);
            accR = __builtin_amdgcn_mfma_f32_16x16x32_bf16(urm, xrm, accR, 0, 0, 0);
            accT = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uim, xim, accT, 0, 0, 0);
            accI = __builtin_amdgcn_mfma_f32_16x16x32_bf16(urm, xim, accI, 0, 0, 0);
            accJ = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uim, xrm, accJ, 0, 0, 0);
            accR = __builtin_amdgcn_mfma_f32_16x16x32_bf16(urh, xrm, accR, 0, 0, 0);
            accT = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uih, xim, accT, 0, 0, 0);
            accI = __builtin_amdgcn_mfma_f32_16x16x32_bf16(urh, xim, accI, 0, 0, 0);
            accJ = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uih, xrm, accJ, 0, 0, 0);
            accR = __builtin_amdgcn_mfma_f32_16x16x32_bf16(urm, xrh, accR, 0, 0, 0);
            accT = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uim, xih, accT, 0, 0, 0);
            accI = __builtin_amdgcn_mfma_f32_16x16x32_bf16(urm, xih, accI, 0, 0, 0);
            accJ = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uim, xrh, accJ, 0, 0, 0);
            accR = __builtin_amdgcn_mfma_f32_16x16x32_bf16(urh, xrh, accR, 0, 0, 0);
            accT = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uih, xih, accT, 0, 0, 0);
            accI = __builtin_amdgcn_mfma_f32_16x16x32_bf16(urh, xih, accI, 0, 0, 0);
            accJ = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uih, xrh, accJ, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i)
              ys[roff(4 * rb + i) ^ tc[w]] =
                  make_float2(flip_sign(accR[i] - accT[i], fl), flip_sign(accI[i] + accJ[i], fl));
          }
        }
        continue;
      }
      bf8 xrh[CBW], xrl[CBW], xih[CBW], xil[CBW];
#pragma unroll
      for (int w = 0; w < CBW; ++w) {
        float2 v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = ys[roff(e) ^ tc[w]];
        split_bf8(v, &xrh[w], &xrl[w], &xih[w], &xil[w]);
      }
      // a row block's U fragments are read (once for all the wave's column
      // blocks) just before its products; the second block's reads are
      // issued before the first block's results are written
      bf8 urh, url, uih, uil;
      if constexpr (U_DIRECT) {
        urh = Af[0][0], url = Af[0][1], uih = Af[0][2], uil = Af[0][3];
      } else {
        urh = As[0], url = As[64], uih = As[128], uil = As[192];
      }
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) {
        // Re = Ur Xr - Ui Xi, Im = Ur Xi + Ui Xr, each real product as
        // hi*hi + hi*lo + lo*hi: four independent chains of three per block
        v4f_t accR[CBW], accT[CBW], accI[CBW], accJ[CBW];
#pragma unroll
        for (int w = 0; w < CBW; ++w) {
          const v4f_t z = {0, 0, 0, 0};
          accR[w] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(urh, xrh[w], z, 0, 0, 0);
          accT[w] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uih, xih[w], z, 0, 0, 0);
          accI[w] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(urh, xih[w], z, 0, 0, 0);
          accJ[w] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uih, xrh[w], z, 0, 0, 0);
        }
#pragma unroll
        for (int w = 0; w < CBW; ++w) {
          accR[w] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(urh, xrl[w], accR[w], 0, 0, 0);
          accT[w] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uih, xil[w], accT[w], 0, 0, 0);
          accI[w] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(urh, xil[w], accI[w], 0, 0, 0);
          accJ[w] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uih, xrl[w], accJ[w], 0, 0, 0);
        }
#pragma unroll
        for (int w = 0; w < CBW; ++w) {
          accR[w] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(url, xrh[w], accR[w], 0, 0, 0);
          accT[w] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uil, xih[w], accT[w], 0, 0, 0);
          accI[w] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(url, xih[w], accI[w], 0, 0, 0);
          accJ[w] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uil, xrh[w], accJ[w], 0, 0, 0);
        }
        if (rb == 0) {
          if constexpr (U_DIRECT) {
            urh = Af[1][0], url = Af[1][1], uih = Af[1][2], uil = Af[1][3];
          } else {
            urh = As[256], url = As[320], uih = As[384], uil = As[448];
          }
        }
        // every wave has read its rows of this step above: write in place
#pragma unroll
        for (int w = 0; w < CBW; ++w)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            ys[roff(4 * rb + i) ^ tc[w]] = make_float2(accR[w][i] - accT[w][i], accI[w][i] + accJ[w][i]);
      }
    }
    __syncthreads();
#pragma unroll 8
    for (int j = 0; j < PER; ++j) {
      const int t = p_lo | phi[wave + W * j];
      const float2 y = ys[t ^ swz[t >> 4]];
      V o;
      o.x = (R)y.x;
      o.y = (R)y.y;
      st_stream<R>(&a[base + a_lo + ahi[wave + W * j]], o);
    }
  }
}

// ---- step grouping on the device ---------------------------------------------
// step_groups (partition.cpp), the beam search over the k-subsets of a wide
// part's qubits that cuts its gates into the fewest fused steps, for all parts
// of a call at once, with the same choices (extensions in the order of gates
// left, state, subset; equal sets of gates left kept once). On the host it
// takes 2 to 5 ms a part, several times the pass itself below 29 qubits. Each
// level of the search is two launches: k_plan_score scores every (part, state,
// subset), a wave 64 subsets of one state, over the whole chip; k_plan_select,
// one workgroup per part and a wave per state, keeps the level's best. Bound by
// the serial chain of levels and, in it, of kept extensions: for the 10 parts
// of a 27-qubit QFT (12 levels) 8 to 15 us a score and 40 to 80 us a
// selection, 0.9 ms in all. With one wave going through all states' extensions
// and absorbing them again a selection took 200 to 700 us; all levels in one
// workgroup per part, on 10 of the 256 CUs, 2.5 ms. The whole pass at 27
// qubits: 34.1 -> 13.8 ms (11.5 with the steps' matrices from the device too).
constexpr int kPlanGates = 128;   // gates of a part, at most (two 64-bit masks)
constexpr int kPlanQubits = 14;
constexpr int kPlanSubsets = 2002;  // C(14, 5)
constexpr int kPlanStride = 2048;
constexpr int kPlanWidth = 16;
constexpr int kPlanLevels = 24;     // steps of a part, at most
constexpr int kPlanThreads = 256;
constexpr size_t kPlanParts = 64;   // parts searched at once (their states are 37 MB)
constexpr double kPlanWork = 12500;  // subsets times gates from which the device is asked

struct PlanPart {
  int num_gates, num_qubits;
  int masks;    // its first gate mask
  int out;      // its answer: the number of groups, then their qubit sets (0 groups: not found)
};

// A part's search, in device memory.
struct PlanState {
  uint64_t rem[2][kPlanWidth][2];   // per state of a level: the gates left
  uint64_t on[kPlanQubits][2];      // the gates on each qubit
  int states, done;
  uint32_t seen[8];                 // numbers of gates left that occur in the level
  uint16_t set[kPlanLevels][kPlanWidth];
  uint8_t parent[kPlanLevels][kPlanWidth];
  uint16_t sub[kPlanStride];        // the subsets, lexicographic by ascending elements
  // gates left after the extension of state b by subset q, at b * kPlanStride
  // + q (255: it takes none)
  alignas(16) uint8_t left[kPlanWidth * kPlanStride];
  uint64_t keep[kPlanWidth * kPlanStride][2];  // the gates it leaves
};

__host__ __device__ constexpr int binomial(int n, int k) {
  if (k < 0 || k > n) return 0;
  int c = 1;
  for (int i = 0; i < k; ++i) c = c * (n - i) / (i + 1);
  return c;
}

// The gates of `rem` (two words) that the blocking scan of the qubit set Q
// takes: those inside Q that share no qubit with an earlier skipped one. on[x]:
// the gates on qubit x. The skipped ones grow from the gates that leave Q: on
// each qubit of Q everything from its first skipped gate on, until no qubit
// adds any (v | -v: the bits from v's lowest up). WIDE: more than 64 gates.
template <bool WIDE>
__device__ __forceinline__ void plan_absorb(uint64_t rem0, uint64_t rem1, const uint64_t (*on)[2], int n, uint32_t Q,
                                            uint64_t* take0, uint64_t* take1) {
  uint64_t s0 = 0, s1 = 0;
  for (int x = 0; x < n; ++x) {
    const uint64_t out = (Q >> x & 1) ? 0 : ~0ull;
    s0 |= on[x][0] & out;
    if constexpr (WIDE) s1 |= on[x][1] & out;
  }
  s0 &= rem0;
  s1 &= rem1;
  uint64_t q0[5], q1[5];
  uint32_t rest = Q;
#pragma unroll
  for (int i = 0; i < 5; ++i) {  // fewer than five: qubit 0's gates of none
    const int x = rest ? __builtin_ctz(rest) : 0;
    q0[i] = rest ? on[x][0] & rem0 : 0;
    q1[i] = WIDE && rest ? on[x][1] & rem1 : 0;
    rest &= rest - 1;
  }
  for (;;) {
    uint64_t a0 = s0, a1 = s1;
#pragma unroll
    for (int i = 0; i < 5; ++i) {
      const uint64_t v0 = a0 & q0[i], n0 = 0 - v0;
      a0 |= q0[i] & (v0 | n0);
      if constexpr (WIDE) {
        const uint64_t v1 = a1 & q1[i];
        a1 |= q1[i] & (v0 ? ~0ull : v1 | (0 - v1));
      }
    }
    const bool more = a0 != s0 || (WIDE && a1 != s1);
    s0 = a0;
    s1 = a1;
    if (!__ballot(more)) break;
  }
  *take0 = rem0 & ~s0;
  *take1 = WIDE ? rem1 & ~s1 : 0;
}

__device__ __forceinline__ uint64_t uniform64(uint64_t x) {
  return uint64_t(uint32_t(__builtin_amdgcn_readfirstlane((int)uint32_t(x)))) |
         uint64_t(uint32_t(__builtin_amdgcn_readfirstlane((int)uint32_t(x >> 32)))) << 32;
}

__global__ __launch_bounds__(kPlanThreads) void k_plan_start(const PlanPart* __restrict__ parts,
                                                             const uint16_t* __restrict__ masks, int k,
                                                             PlanState* __restrict__ states, uint16_t* __restrict__ out) {
  const PlanPart P = parts[blockIdx.x];
  PlanState& S = states[blockIdx.x];
  const int n = P.num_qubits, kk = k < n ? k : n, ns = binomial(n, kk), ng = P.num_gates;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int q = threadIdx.x; q < ns; q += kPlanThreads) {
    int r = q, x = 0;
    uint32_t c = 0;
    for (int i = 0; i < kk; ++i, ++x) {
      for (int b; r >= (b = binomial(n - 1 - x, kk - 1 - i)); ++x) r -= b;
      c |= 1u << x;
    }
    S.sub[q] = (uint16_t)c;
  }
  for (int x = wave; x < 2 * n; x += kPlanThreads / 64) {
    const int i = 64 * (x & 1) + lane;
    const uint64_t g = __ballot(i < ng && (masks[P.masks + i] >> (x >> 1) & 1));
    if (lane == 0) S.on[x >> 1][x & 1] = g;
  }
  if (threadIdx.x < 8) S.seen[threadIdx.x] = 0;
  if (threadIdx.x == 0) {
    S.rem[0][0][0] = ng >= 64 ? ~0ull : (1ull << ng) - 1;
    S.rem[0][0][1] = ng <= 64 ? 0 : ng == 128 ? ~0ull : (1ull << (ng - 64)) - 1;
    S.states = 1;
    S.done = 0;
    out[P.out] = 0;
  }
}

// Level `level` of part blockIdx.y: state blockIdx.z, 256 subsets a block.
__global__ __launch_bounds__(kPlanThreads) void k_plan_score(const PlanPart* __restrict__ parts, int k, int level,
                                                             PlanState* __restrict__ states) {
  const PlanPart P = parts[blockIdx.y];
  PlanState& S = states[blockIdx.y];
  const int b = blockIdx.z, n = P.num_qubits, kk = k < n ? k : n, ns = binomial(n, kk);
  if (S.done || b >= S.states || (int)blockIdx.x * kPlanThreads >= ns) return;  // uniform
  __shared__ uint64_t on[kPlanQubits][2];
  if (threadIdx.x < 2 * n) on[threadIdx.x >> 1][threadIdx.x & 1] = S.on[threadIdx.x >> 1][threadIdx.x & 1];
  __syncthreads();
  const int q = blockIdx.x * kPlanThreads + threadIdx.x;
  const uint64_t r0 = uniform64(S.rem[level & 1][b][0]), r1 = uniform64(S.rem[level & 1][b][1]);
  const uint32_t Q = q < ns ? S.sub[q] : 0;
  uint64_t t0, t1;
  if (r1) plan_absorb<true>(r0, r1, on, n, Q, &t0, &t1);
  else plan_absorb<false>(r0, r1, on, n, Q, &t0, &t1);
  const int got = __popcll(t0) + __popcll(t1);
  const int l = q < ns && got > 0 ? __popcll(r0) + __popcll(r1) - got : 255;
  S.left[b * kPlanStride + q] = (uint8_t)l;
  S.keep[b * kPlanStride + q][0] = r0 & ~t0;
  S.keep[b * kPlanStride + q][1] = r1 & ~t1;
  // one atomic per word and wave
  for (int w = 0; w < 8; ++w) {
    uint32_t bits = (l >> 5) == w ? 1u << (l & 31) : 0;
    for (int m = 32; m >= 1; m >>= 1) bits |= __shfl_xor(bits, m);
    if ((threadIdx.x & 63) == 0 && bits) atomicOr(&S.seen[w], bits);
  }
}

// Keeps the best kPlanWidth extensions of a level, wave b going through state
// b's: for each number of gates left, from the lowest, the waves list their
// state's first distinct extensions (kPlanWidth of them are enough: each one
// that the states before have already is one of the kept), and the first wave
// takes them in order, those whose gates left are new.
constexpr int kPlanSelect = 64 * kPlanWidth;
__global__ __launch_bounds__(kPlanSelect) void k_plan_select(const PlanPart* __restrict__ parts, int k, int level,
                                                             PlanState* __restrict__ states,
                                                             uint16_t* __restrict__ out) {
  const PlanPart P = parts[blockIdx.x];
  PlanState& S = states[blockIdx.x];
  if (S.done) return;  // uniform
  const int n = P.num_qubits, kk = k < n ? k : n, ns = binomial(n, kk), now = level & 1, nstates = S.states;
  __shared__ __align__(16) uint8_t left[kPlanWidth * kPlanStride];
  __shared__ uint64_t list[kPlanWidth][kPlanWidth][2];
  __shared__ uint16_t list_q[kPlanWidth][kPlanWidth];
  __shared__ int listed[kPlanWidth], taken_sh;
  const int rows = (ns + 255) / 256;  // 256-byte rows that were scored, per state
  for (int i = threadIdx.x; i < nstates * rows * 16; i += kPlanSelect) {
    const int b = i / (rows * 16), o = b * kPlanStride + (i - b * rows * 16) * 16;
    *reinterpret_cast<uint4*>(left + o) = *reinterpret_cast<const uint4*>(S.left + o);
  }
  uint32_t seen[8];
#pragma unroll
  for (int w = 0; w < 8; ++w) seen[w] = S.seen[w];
  const int lane = threadIdx.x & 63, b = threadIdx.x >> 6;
  int taken = 0;
  uint64_t kept0 = 0, kept1 = 0;  // first wave, lane j: the gates left of the j-th kept extension
  __syncthreads();  // left; every thread has read seen
  if (threadIdx.x < 8) S.seen[threadIdx.x] = 0;
  for (int v = 0; v < 255 && taken < kPlanWidth; ++v) {
    if (!(seen[v >> 5] >> (v & 31) & 1)) continue;  // uniform
    int mine = 0;
    uint64_t own0 = 0, own1 = 0;
    int own_q = 0;
    for (int q0 = 0; b < nstates && q0 < ns && mine < kPlanWidth; q0 += 256) {
      // four numbers a lane: which of the 256 are v
      const uint32_t w = *reinterpret_cast<const uint32_t*>(left + b * kPlanStride + q0 + 4 * lane);
      const bool any = (w & 255u) == (uint32_t)v || (w >> 8 & 255u) == (uint32_t)v || (w >> 16 & 255u) == (uint32_t)v ||
                       w >> 24 == (uint32_t)v;
      const uint64_t quads = __ballot(any);
      for (int c = 0; c < 4 && mine < kPlanWidth; ++c) {
        if (!(quads >> (16 * c) & 0xffffu)) continue;
        const int q = q0 + 64 * c + lane;
        uint64_t hits = __ballot(left[b * kPlanStride + q] == (uint8_t)v);
        const uint64_t k0 = S.keep[b * kPlanStride + q][0], k1 = S.keep[b * kPlanStride + q][1];
        while (hits && mine < kPlanWidth) {
          const int h = __builtin_ctzll(hits);
          const uint64_t h0 = uint64_t(uint32_t(__builtin_amdgcn_readlane((int)uint32_t(k0), h))) |
                              uint64_t(uint32_t(__builtin_amdgcn_readlane((int)uint32_t(k0 >> 32), h))) << 32;
          const uint64_t h1 = uint64_t(uint32_t(__builtin_amdgcn_readlane((int)uint32_t(k1), h))) |
                              uint64_t(uint32_t(__builtin_amdgcn_readlane((int)uint32_t(k1 >> 32), h))) << 32;
          hits &= ~__ballot(k0 == h0 && k1 == h1);  // with it the others that leave the same gates
          if (__ballot(lane < mine && own0 == h0 && own1 == h1)) continue;
          if (lane == mine) {
            own0 = h0;
            own1 = h1;
            own_q = q0 + 64 * c + h;
          }
          ++mine;
        }
      }
    }
    if (lane < mine) {
      list[b][lane][0] = own0;
      list[b][lane][1] = own1;
      list_q[b][lane] = (uint16_t)own_q;
    }
    if (lane == 0) listed[b] = mine;
    __syncthreads();
    if (v == 0) {  // a state without gates left: the search ends with its first
      if (threadIdx.x == 0) {
        int x = 0;
        while (!listed[x]) ++x;
        uint16_t* o = out + P.out;
        o[0] = (uint16_t)(level + 1);
        o[1 + level] = S.sub[list_q[x][0]];
        for (int at = level - 1; at >= 0; --at) {
          o[1 + at] = S.set[at][x];
          x = S.parent[at][x];
        }
        S.done = 1;
      }
      return;
    }
    if (b == 0) {
      for (int x = 0; x < nstates && taken < kPlanWidth; ++x) {
        const int cnt = listed[x];
        const uint64_t k0 = lane < cnt ? list[x][lane][0] : 0, k1 = lane < cnt ? list[x][lane][1] : 0;
        for (int h = 0; h < cnt && taken < kPlanWidth; ++h) {
          const uint64_t h0 = uint64_t(uint32_t(__builtin_amdgcn_readlane((int)uint32_t(k0), h))) |
                              uint64_t(uint32_t(__builtin_amdgcn_readlane((int)uint32_t(k0 >> 32), h))) << 32;
          const uint64_t h1 = uint64_t(uint32_t(__builtin_amdgcn_readlane((int)uint32_t(k1), h))) |
                              uint64_t(uint32_t(__builtin_amdgcn_readlane((int)uint32_t(k1 >> 32), h))) << 32;
          if (__ballot(lane < taken && kept0 == h0 && kept1 == h1)) continue;
          if (lane == taken) {
            kept0 = h0;
            kept1 = h1;
            S.parent[level][taken] = (uint8_t)x;
            S.set[level][taken] = S.sub[list_q[x][h]];
          }
          ++taken;
        }
      }
      if (lane == 0) taken_sh = taken;
    }
    __syncthreads();  // the lists are read
    taken = taken_sh;
  }
  if (b == 0) {
    if (lane < taken) {
      S.rem[now ^ 1][lane][0] = kept0;
      S.rem[now ^ 1][lane][1] = kept1;
    }
    if (lane == 0) {
      S.states = taken;
      if (!taken) S.done = 1;  // no gate fits: the host reports it
    }
  }
}

// ---- the steps' matrices on the device -----------------------------------------
// What the host does otherwise before each pass, 0.3 to 0.9 ms a part: 28 us a
// step for the check that its matrix is unitary, 7 us for its BF16 fragments,
// up to 0.4 ms for the part's swizzle. For all parts at once instead: 13 and 24
// us for the 65 steps of a 27-qubit QFT, bound by latency (one workgroup a
// step, a part).
__host__ __device__ inline uint16_t bf16_bits(float f) {
  // round to nearest even (finite inputs; NaN stays NaN)
  uint32_t u;
  __builtin_memcpy(&u, &f, 4);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__host__ __device__ inline double bf16_value(uint16_t h) {
  const uint32_t u = (uint32_t)h << 16;
  float f;
  __builtin_memcpy(&f, &u, 4);
  return f;
}
// The BF16 fragments of a step's matrix in the MFMA's A-operand order: entry e
// of lane `lane` in row block rb is U[part_bf_row][part_bf_col]; its pieces are
// 64 * 8 apart, the real ones first.
__host__ __device__ inline int part_bf_row(int rb, int lane) {
  const int mm = lane % 16;
  return 16 * rb + 4 * (mm % 4) + mm / 4;
}
__host__ __device__ inline int part_bf_col(int lane, int e) { return lane / 16 + 4 * e; }
__host__ __device__ inline void part_bf_pieces(double re, double im, int pieces, uint16_t* frag) {
  // each piece the BF16 of what the previous ones leave of the FP64 entry
  for (int k = 0; k < pieces; ++k) {
    const uint16_t pr = bf16_bits((float)re), pi = bf16_bits((float)im);
    frag[size_t(k) * 64 * 8] = pr;
    frag[size_t(pieces + k) * 64 * 8] = pi;
    re -= bf16_value(pr);
    im -= bf16_value(pi);
  }
}

// One workgroup per step. uerr: max |U^H U - I|, a NaN left out as in
// unitarity_error; -1 when an entry is not finite or huge (the host
// then decides).
constexpr int kStepThreads = 256;
__global__ __launch_bounds__(kStepThreads) void k_part_steps(const double2* __restrict__ U, int pieces,
                                                             uint16_t* __restrict__ frags, double* __restrict__ uerr) {
  __shared__ double2 u[32 * 32];
  __shared__ double worst[kStepThreads];
  __shared__ int bad;
  const int t = threadIdx.x;
  if (t == 0) bad = 0;
  __syncthreads();
  for (int i = t; i < 32 * 32; i += kStepThreads) {
    u[i] = U[size_t(blockIdx.x) * 1024 + i];
    if (!(fabs(u[i].x) < 1e100 && fabs(u[i].y) < 1e100)) bad = 1;
  }
  __syncthreads();
  double w = 0;
  for (int p = t; p < 32 * 32; p += kStepThreads) {
    const int i = p >> 5, j = p & 31;
    double x = 0, y = 0;
    for (int r = 0; r < 32; ++r) {
      const double2 a = u[r * 32 + i], b = u[r * 32 + j];
      x += a.x * b.x + a.y * b.y;
      y += a.x * b.y - a.y * b.x;
    }
    if (i == j) x -= 1.0;
    w = fmax(w, sqrt(x * x + y * y));
  }
  worst[t] = w;
  __syncthreads();
  for (int h = kStepThreads / 2; h; h >>= 1) {
    if (t < h) worst[t] = fmax(worst[t], worst[t + h]);
    __syncthreads();
  }
  if (t == 0) uerr[blockIdx.x] = bad ? -1.0 : worst[0];
  uint16_t* f = frags + size_t(blockIdx.x) * 2 * 2 * pieces * 64 * 8;
  for (int i = t; i < 2 * 64 * 8; i += kStepThreads) {
    const int e = i & 7, lane = i >> 3 & 63, rb = i >> 9;
    const double2 v = u[part_bf_row(rb, lane) * 32 + part_bf_col(lane, e)];
    part_bf_pieces(v.x, v.y, pieces, f + (size_t(rb) * 2 * pieces * 64 + lane) * 8 + e);
  }
}

// The LDS swizzle of a part (choose_part_swizzle, with the same choice): its
// 2000 candidates over the threads of a workgroup, each thread two that follow
// each other in the generator's sequence, from its state before them.
struct PartSwizzleKey { int cbit[4]; int rbit0; };
struct SwizzlePart {
  int KT, first, count;  // its keys
};
constexpr int kSwizzleTries = 2000, kSwizzleThreads = 1024, kSwizzleEach = 2;
static_assert(kSwizzleThreads * kSwizzleEach >= kSwizzleTries, "a thread for each candidate");
__host__ __device__ inline void swizzle_candidate(uint64_t* rng, int KT, uint32_t* cand) {
  uint64_t r = *rng;
  for (int c = 0; c < 14; ++c) {
    r ^= r << 13;
    r ^= r >> 7;
    r ^= r << 17;
    cand[c] = c < 4 ? 0u : (c == 4 ? uint32_t(r & 15u) : (c < KT ? uint32_t(r & 31u) : 0u));
  }
  *rng = r;
}
__global__ __launch_bounds__(kSwizzleThreads) void k_part_swizzle(const SwizzlePart* __restrict__ parts,
                                                                  const PartSwizzleKey* __restrict__ keys,
                                                                  const uint64_t* __restrict__ rng,
                                                                  uint32_t* __restrict__ nimg) {
  const SwizzlePart P = parts[blockIdx.x];
  __shared__ uint32_t img[14][kSwizzleThreads + 1];  // a thread's candidate: a column
  __shared__ int best[kSwizzleThreads];              // score * 4096 + 4095 - (its place in the sequence)
  const int t = threadIdx.x;
  int mine = -1;
  uint64_t r = t * kSwizzleEach < kSwizzleTries ? rng[t] : 0;
  // the sequence: no swizzle at all, then the candidates
  for (int e = -1; e < kSwizzleEach; ++e) {
    if (e < 0 ? t != 0 : t * kSwizzleEach + e >= kSwizzleTries) continue;
    uint32_t cand[14] = {0};
    if (e >= 0) swizzle_candidate(&r, P.KT, cand);
#pragma unroll
    for (int c = 0; c < 14; ++c) img[c][t] = (c < 5 ? 1u << c : 0u) ^ cand[c];
    int sc = 0;
    for (int k = P.first; k < P.first + P.count; ++k) {
      uint32_t v[5];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = img[keys[k].cbit[j]][t];
      v[4] = img[keys[k].rbit0][t];
      // independent: no sum of some of them is 0
      uint32_t sum[32];
      bool four = true, five = true;
      sum[0] = 0;
#pragma unroll
      for (int m = 1; m < 32; ++m) {
        sum[m] = sum[m & (m - 1)] ^ v[__builtin_ctz(m)];
        five = five && (sum[m] & 31u);
        if (m < 16) four = four && (sum[m] & 15u);
      }
      sc += 2 * four + five;
    }
    mine = max(mine, sc * 4096 + 4095 - (t * kSwizzleEach + e + 1));
  }
  best[t] = mine;
  __syncthreads();
  for (int h = kSwizzleThreads / 2; h; h >>= 1) {
    if (t < h) best[t] = max(best[t], best[t + h]);
    __syncthreads();
  }
  if (t == 0) {
    const int at = 4095 - (best[0] & 4095) - 1;  // -1: no swizzle
    uint32_t cand[14] = {0};
    if (at >= 0) {
      uint64_t q = rng[at / kSwizzleEach];
      for (int e = 0; e <= at % kSwizzleEach; ++e) swizzle_candidate(&q, P.KT, cand);
    }
    for (int c = 0; c < 14; ++c) nimg[blockIdx.x * 14 + c] = cand[c];
  }
}

namespace {

// the highest `count` slots of an outer mask (the tile kernels' fast slots)
uint64_t top_slots(uint64_t outer, int count) {
  uint64_t top = 0;
  for (int i = 0; i < count && (outer & ~top); ++i) top |= 1ull << (63 - __builtin_clzll(outer & ~top));
  return top;
}

uint64_t pdep_host(uint64_t x, uint64_t mask) {
  uint64_t r = 0;
  for (uint64_t bit = 1; mask; bit <<= 1) {
    const uint64_t low = mask & (~mask + 1);
    if (x & bit) r |= low;
    mask &= mask - 1;
  }
  return r;
}

template <typename R, int K, bool SPLIT>
void launch(void* amp, const void* scratch, int D, int C, int grid, hipStream_t st, const FusedArgs& f) {
  const double2* U = static_cast<const double2*>(scratch);
  const uint64_t* qoff = reinterpret_cast<const uint64_t*>(U + size_t(D) * D);
  const uint64_t* toff = qoff + D;
  const size_t lds = size_t(D) * C * sizeof(double2);
  hipLaunchKernelGGL((k_fused<R, K, SPLIT>), grid, 4 * (1 << K), lds, st,
                     static_cast<typename VecT<R>::type*>(amp), U, qoff, toff, f);
}

template <typename R, bool SPLIT>
void launch_k(int K, void* amp, const void* scratch, int D, int C, int grid, hipStream_t st, const FusedArgs& f) {
  switch (K) {
    case 4: launch<R, 4, SPLIT>(amp, scratch, D, C, grid, st, f); break;
    case 5: launch<R, 5, SPLIT>(amp, scratch, D, C, grid, st, f); break;
    case 6: launch<R, 6, SPLIT>(amp, scratch, D, C, grid, st, f); break;
    default: launch<R, 7, SPLIT>(amp, scratch, D, C, grid, st, f); break;
  }
}

}  // namespace

int fused_unitary(int n, const std::vector<Lowered>& gates, std::vector<int>* qubits, std::vector<cd>* U,
                  std::string* err, int min_qubits) {
  uint64_t mask = 0;
  for (const Lowered& L : gates) {
    for (int i = 0; i < L.nt; ++i) mask |= 1ull << L.t[i];
    for (int i = 0; i < L.nc; ++i) mask |= 1ull << L.c[i];
  }
  if (__builtin_popcountll(mask) > 7) {
    *err = "fused parts take at most 7 qubits";
    return HSV_ERR_LIMIT;
  }
  if (n < min_qubits) {
    *err = "fused parts need at least " + std::to_string(min_qubits) + " qubits in the state";
    return HSV_ERR_LIMIT;
  }
  for (int b = 0; b < n && __builtin_popcountll(mask) < min_qubits; ++b) mask |= 1ull << b;  // pad: U (x) I
  qubits->clear();
  for (int b = 0; b < 64; ++b)
    if (mask >> b & 1) qubits->push_back(b);
  build_fused(gates, *qubits, U);
  return HSV_OK;
}

namespace {

int ensure_scratch(DeviceScratch* scratch, size_t bytes, hipStream_t stream, std::string* err) {
  if (scratch->bytes >= bytes) return HSV_OK;
  if (scratch->fixed) {
    *err = "this part needs " + std::to_string(bytes) + " bytes of device scratch; the no-allocation entry point "
           "has " + std::to_string(scratch->bytes);
    return HSV_ERR_LIMIT;
  }
  if (hipStreamSynchronize(stream) != hipSuccess) { *err = "stream sync failed"; return HSV_ERR_DEVICE; }
  if (scratch->ptr) (void)hipFree(scratch->ptr);
  scratch->ptr = nullptr;
  scratch->bytes = 0;
  const size_t cap = std::max<size_t>(bytes, 1 << 20);
  if (hipMalloc(&scratch->ptr, cap) != hipSuccess) { *err = "fused scratch allocation failed"; return HSV_ERR_ALLOC; }
  scratch->bytes = cap;
  return HSV_OK;
}

template <typename R, int K, bool SWZ>
void launch_bf(void* amp, const void* scratch, int grid, hipStream_t st, const BfArgs& f, int* rc) {
  constexpr int D = 1 << K;
  const size_t frag_bytes = size_t(8) * D * D;
  const auto* U = static_cast<const bf8*>(scratch);
  const uint64_t* qoff = reinterpret_cast<const uint64_t*>(static_cast<const unsigned char*>(scratch) + frag_bytes);
  const uint64_t* toff = qoff + D;
  auto kern = &k_fused_bf<R, K, SWZ>;
  if (frag_bytes > 65536 &&
      hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int)frag_bytes) != hipSuccess) {
    *rc = HSV_ERR_DEVICE;
    return;
  }
  hipLaunchKernelGGL(kern, grid, kBfThreads, frag_bytes, st, static_cast<typename VecT<R>::type*>(amp), U, qoff,
                     toff, f);
}

// The BF16-split path: U as BF16 hi/lo fragments in the MFMA A-operand order,
// columns in blocks of 16 along the lowest 4 slots outside the part.
template <typename R, int K>
void launch_bft(void* amp, const void* scratch, int grid, hipStream_t st, uint64_t ntiles, uint64_t outer, uint64_t top,
                int tpw) {
  const size_t frag_bytes = size_t(8) << (2 * K);
  const auto* U = static_cast<const bf8*>(scratch);
  const auto* T = reinterpret_cast<const BfTileTables*>(static_cast<const unsigned char*>(scratch) + frag_bytes);
  hipLaunchKernelGGL((k_fused_bft<R, K>), grid, kBfTileThreads, 0, st,
                     static_cast<typename VecT<R>::type*>(amp), U, T, ntiles, outer, top, tpw);
}

// Tables of the tile form: tile index bit j <-> the j-th lowest of the tile's
// 12 slots (the part's qubits plus the 12 - K lowest slots outside it).
void build_tile_tables(uint64_t qmask, uint64_t cmask, BfTileTables* T) {
  int slot[12], rowpos[12], colpos[12];
  int j = 0, nr = 0, nc = 0;
  for (int b = 0; b < 64 && j < 12; ++b) {
    if (qmask >> b & 1) { slot[j] = b; rowpos[j] = nr++; colpos[j] = -1; ++j; }
    else if (cmask >> b & 1) { slot[j] = b; rowpos[j] = -1; colpos[j] = nc++; ++j; }
  }
  std::memset(T, 0, sizeof(*T));
  for (int v = 0; v < 64; ++v)
    for (int bit = 0; bit < 6; ++bit) {
      if (!(v >> bit & 1)) continue;
      T->alo[v] += 1ull << slot[bit];
      T->ahi[v] += 1ull << slot[6 + bit];
      if (rowpos[bit] >= 0) T->rlo[v] += (uint16_t)(1u << rowpos[bit]);
      if (rowpos[6 + bit] >= 0) T->rhi[v] += (uint16_t)(1u << rowpos[6 + bit]);
      if (colpos[bit] >= 0) T->clo[v] += (uint16_t)(1u << colpos[bit]);
      if (colpos[6 + bit] >= 0) T->chi[v] += (uint16_t)(1u << colpos[6 + bit]);
    }
  for (int q = 0; q < 12; ++q) {
    for (int r = 0; r < (1 << nr); ++r)
      if (rowpos[q] >= 0 && (r >> rowpos[q] & 1)) T->tr[r] |= (uint16_t)(1u << q);
    for (int c = 0; c < (1 << nc); ++c)
      if (colpos[q] >= 0 && (c >> colpos[q] & 1)) T->tc[c] |= (uint16_t)(1u << q);
  }
}

// LDS swizzle of k_part_bf. nimg[c] = h applied to tile bit c: 0 for
// c < 4, a mask of bits 0-3 for c = 4, of bits 0-4 for c >= 5. A step is
// conflict-free when the low-4-bit images of its 4 lowest column bits are
// independent (the 16 lanes of a quarter-wave) and, with its lowest row bit,
// the low-5-bit images are too (the 32 lanes of a half-wave).
// rank over GF(2) of n <= 5 vectors of 5 bits
int rank_gf2(uint32_t* v, int n) {
  int r = 0;
  for (int bit = 4; bit >= 0; --bit) {
    int piv = -1;
    for (int i = r; i < n; ++i)
      if (v[i] >> bit & 1) { piv = i; break; }
    if (piv < 0) continue;
    std::swap(v[r], v[piv]);
    for (int i = 0; i < n; ++i)
      if (i != r && (v[i] >> bit & 1)) v[i] ^= v[r];
    ++r;
  }
  return r;
}

constexpr uint64_t kSwizzleSeed = 0x9E3779B97F4A7C15ull;

void choose_part_swizzle(int KT, const std::vector<PartSwizzleKey>& keys, uint32_t nimg[14]) {
  int best = -1;
  auto score = [&](const uint32_t* m) {
    int sc = 0, open = 3 * (int)keys.size();
    for (const PartSwizzleKey& k : keys) {
      if (sc + open <= best) return sc;  // cannot become the best any more
      open -= 3;
      auto low5 = [&](int c) { return ((c < 5) ? (1u << c) : 0u) ^ m[c]; };
      uint32_t a[4], b[5];
      for (int j = 0; j < 4; ++j) { b[j] = low5(k.cbit[j]); a[j] = b[j] & 15u; }
      b[4] = low5(k.rbit0);
      sc += 2 * (rank_gf2(a, 4) == 4) + (rank_gf2(b, 5) == 5);
    }
    return sc;
  };
  const int best_possible = 3 * (int)keys.size();
  uint32_t cand[14] = {0};
  std::memcpy(nimg, cand, sizeof(cand));
  best = score(cand);
  uint64_t rng = kSwizzleSeed;
  for (int it = 0; it < kSwizzleTries && best < best_possible; ++it) {
    swizzle_candidate(&rng, KT, cand);
    const int sc = score(cand);
    if (sc > best) { best = sc; std::memcpy(nimg, cand, sizeof(cand)); }
  }
}

template <typename R, int KT, bool STREAM_U, bool U_DIRECT = false, int NP = 2>
void launch_part_bf(void* amp, const unsigned char* dev, size_t tabs_off, size_t steps_off, size_t frag_off,
                    int nsteps, int grid, hipStream_t st, uint64_t ntiles, uint64_t outer, uint64_t top, int tpw,
                    int* rc) {
  const size_t lds = STREAM_U ? 0 : size_t(nsteps) * 2 * 2 * NP * 64 * sizeof(bf8);
  auto kern = &k_part_bf<R, KT, STREAM_U, U_DIRECT, NP>;
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int)std::max<size_t>(lds, 1)) != hipSuccess) {
    *rc = HSV_ERR_DEVICE;
    return;
  }
  hipLaunchKernelGGL(kern, grid, part_bf_threads(KT, STREAM_U), lds, st, static_cast<typename VecT<R>::type*>(amp),
                     reinterpret_cast<const PartBfTables*>(dev + tabs_off),
                     reinterpret_cast<const PartBfStep*>(dev + steps_off),
                     reinterpret_cast<const bf8*>(dev + frag_off), nsteps, ntiles, outer, top, tpw);
}

// fused_part_prepare and fused_part_launch for a part of 8 to 14 qubits (see
// k_part_bf); phys null: logical qubit q sits in slot q, phys_after null: it
// stays there.
int part_prepare_bf(int n, const std::vector<Lowered>& gates, uint64_t tile_qubits, const int* phys,
                    const int* phys_after, int pieces, const std::vector<std::vector<int>>* planned, FusedPart* P,
                    std::string* err) {
  *P = FusedPart();
  int ph[64], pa[64], inv[64];
  for (int q = 0; q < n; ++q) ph[q] = phys ? phys[q] : q;
  for (int q = 0; q < n; ++q) {
    pa[q] = phys_after ? phys_after[q] : ph[q];
    inv[ph[q]] = q;
  }
  uint64_t pmask = 0;
  for (int q = 0; q < n; ++q)
    if (tile_qubits >> q & 1) pmask |= 1ull << ph[q];
  const int K = __builtin_popcountll(pmask);
  // The tile is the part's qubits padded with the lowest free slots. It
  // should hold slots 0-4, so that each wave's loads and stores cover
  // 512-byte runs: a part that fits 12 qubits only without them takes a
  // 13-qubit tile.
  const uint64_t low5 = (1ull << std::min(n, 5)) - 1;
  const int KT = P->KT = std::max(12, std::min(14, __builtin_popcountll(pmask | low5)));
  if (K > 14) {
    *err = "the bf16 fused path takes parts of at most 14 qubits";
    return HSV_ERR_LIMIT;
  }
  if (n < KT) {
    *err = "a wide bf16 fused part needs a state of at least " + std::to_string(KT) + " qubits";
    return HSV_ERR_LIMIT;
  }
  if (pieces == 3 && KT > 13) {
    *err = "the three-piece bf16 split takes parts whose qubits and slots 0-4 fit 13 qubits";
    return HSV_ERR_LIMIT;
  }
  uint64_t tmask = pmask;
  for (int b = 0; b < n && __builtin_popcountll(tmask) < KT; ++b) tmask |= 1ull << b;
  int *slot = P->slot, *sslot = P->sslot;
  uint64_t smask = 0;
  for (int b = 0, j = 0; b < 64 && j < KT; ++b)
    if (tmask >> b & 1) {
      slot[j] = b;
      sslot[j] = pa[inv[b]];
      smask |= 1ull << sslot[j];
      ++j;
    }
  for (int q = 0; q < n; ++q)
    if (!(tmask >> ph[q] & 1) && pa[q] != ph[q]) smask = 0;
  if (smask != tmask) {
    *err = "the layout change moves a qubit into or out of the part's tile";
    return HSV_ERR_ARG;
  }
  auto inner = [&](int q) { return __builtin_popcountll(tmask & ((1ull << ph[q]) - 1)); };
  for (const Lowered& L : gates) {
    if (L.kind == K_IDENT) continue;  // no-ops: their qubits need no tile slot
    for (int i = 0; i < L.nt + L.nc; ++i)
      if (!(tmask >> ph[i < L.nt ? L.t[i] : L.c[i - L.nt]] & 1)) {
        *err = "a gate acts on a qubit outside the part's tile";
        return HSV_ERR_ARG;
      }
  }
  std::vector<uint64_t> qm;
  std::vector<const Lowered*> gl;
  for (const Lowered& L : gates) {
    if (L.kind == K_IDENT) continue;
    uint64_t m = 0;
    for (int i = 0; i < L.nt; ++i) m |= 1ull << inner(L.t[i]);
    for (int i = 0; i < L.nc; ++i) m |= 1ull << inner(L.c[i]);
    qm.push_back(m);
    gl.push_back(&L);
  }
  P->tmask = tmask;
  for (int j = 0; j < KT; ++j) P->moves = P->moves || sslot[j] != slot[j];
  P->nothing = qm.empty() && !P->moves;  // identities only
  if (P->nothing) return HSV_OK;
  // the steps: groups of <= 5 qubits, as few as a beam of 16 finds
  std::vector<std::vector<int>> groups;
  if (!qm.empty()) groups = planned && !planned->empty() ? *planned : step_groups(qm, 5, kPlanWidth);
  if (groups.empty() && !qm.empty()) {
    *err = "a gate acts on more than 5 qubits: the wide bf16 fused path cannot take it";
    return HSV_ERR_LIMIT;
  }
  P->steps.resize(groups.size());
  for (size_t s = 0; s < groups.size(); ++s) {
    FusedPart::Step& S = P->steps[s];
    uint64_t gm = 0;
    std::vector<Lowered> sg;
    for (int i : groups[s]) { gm |= qm[i]; sg.push_back(*gl[i]); }
    for (int b = 0; b < KT && __builtin_popcountll(gm) < 5; ++b) gm |= 1ull << b;  // pad: U (x) I
    std::vector<int> qubits;
    for (int b = 0, r = 0, c = 0; b < KT; ++b) {
      if (gm >> b & 1) { S.rbit[r++] = b; qubits.push_back(inv[slot[b]]); }
      else S.cbit[c++] = b;
    }
    build_fused(sg, qubits, &S.U);
  }
  return HSV_OK;
}

// A part's keys for the swizzle: its steps' columns, and the store gather of a
// layout change, which reads a quarter-wave's 16 positions along load bits
// sig^-1(0..3): its banks count like a step's columns. sig_inv: tile bit j's
// qubit moves to tile bit sig[j] (the tile position of its new slot); store
// position u reads load position sig^-1(u).
std::vector<PartSwizzleKey> part_keys(const FusedPart& P, int* sig_inv) {
  std::vector<PartSwizzleKey> keys;
  for (const FusedPart::Step& S : P.steps)
    keys.push_back(PartSwizzleKey{{S.cbit[0], S.cbit[1], S.cbit[2], S.cbit[3]}, S.rbit[0]});
  for (int j = 0; j < P.KT; ++j)
    for (int k = 0; k < P.KT; ++k)
      if (P.slot[k] == P.sslot[j]) sig_inv[k] = j;
  if (P.moves) keys.push_back(PartSwizzleKey{{sig_inv[0], sig_inv[1], sig_inv[2], sig_inv[3]}, sig_inv[4]});
  return keys;
}

// the tables of a part before its fragments
size_t part_tables_bytes(size_t ns) {
  return (2 * sizeof(PartBfTables) + sizeof(PartBfStep) * ns + 255) & ~size_t(255);
}

int part_launch_bf(void* amp, int n, int dtype, hipStream_t stream, DeviceScratch* scratch, const FusedPart& P,
                   uint64_t live_slots, const BfTune& bf, int pieces, std::string* err) {
  if (P.nothing) return HSV_OK;
  int tpw = bf.part_tpw;
  const int KT = P.KT, ns = (int)P.steps.size();
  const uint64_t tmask = P.tmask;
  const int* slot = P.slot;
  std::vector<PartBfStep> steps(ns);
  const int nsets = 2 * pieces;   // real pieces, then imaginary pieces
  const size_t step_frag_bytes = size_t(2) * nsets * 64 * 16;
  std::vector<uint16_t> frags(P.checked ? 0 : size_t(ns) * 2 * nsets * 64 * 8);
  for (int s = 0; s < ns; ++s) {
    const FusedPart::Step& F = P.steps[s];
    const double uerr = P.checked && P.uerr[s] >= 0 ? P.uerr[s] : unitarity_error(F.U, 32);
    if (!(uerr <= 1e-10)) {
      *err = "fused step matrix is not unitary (max |U^H U - I| = " + std::to_string(uerr) + ")";
      return HSV_ERR_UNITARY;
    }
    PartBfStep& S = steps[s];
    std::memset(&S, 0, sizeof(S));
    for (int r = 0; r < 32; ++r)
      for (int b = 0; b < 5; ++b)
        if (r >> b & 1) S.rt[r] |= (uint16_t)(1u << F.rbit[b]);
    const int ncb = KT - 5;
    for (int v = 0; v < 32; ++v)
      for (int j = 0; j < 5; ++j) {
        if (!(v >> j & 1)) continue;
        if (j < 4 && j < ncb && v < 16) S.ctl[v] |= (uint16_t)(1u << F.cbit[j]);
        if (4 + j < ncb) S.cth[v] |= (uint16_t)(1u << F.cbit[4 + j]);
      }
    for (int rb = 0; rb < 2 && !P.checked; ++rb)
      for (int lane = 0; lane < 64; ++lane)
        for (int e = 0; e < 8; ++e) {
          const cd u = F.U[size_t(part_bf_row(rb, lane)) * 32 + part_bf_col(lane, e)];
          part_bf_pieces(u.real(), u.imag(), pieces, &frags[(size_t((s * 2 + rb) * nsets) * 64 + lane) * 8 + e]);
        }
  }
  // swizzle the steps' LDS offsets (h is linear: XOR of the bits' images)
  int sig_inv[14];
  const std::vector<PartSwizzleKey> keys = part_keys(P, sig_inv);
  uint32_t nimg[14];
  if (P.checked) std::memcpy(nimg, P.nimg, sizeof(nimg));
  else choose_part_swizzle(KT, keys, nimg);
  auto hmap = [&](uint32_t t) {
    uint32_t h = 0;
    for (int c = 4; c < KT; ++c)
      if (t >> c & 1) h ^= nimg[c];
    return h;
  };
  for (PartBfStep& S : steps) {
    for (auto& x : S.rt) x = (uint16_t)(x ^ hmap(x));
    for (auto& x : S.ctl) x = (uint16_t)(x ^ hmap(x));
    for (auto& x : S.cth) x = (uint16_t)(x ^ hmap(x));
  }
  // two table sets: T0 stores where it loads (passes before the last, when
  // the steps need several), T applies the layout change
  PartBfTables T0, T;
  std::memset(&T0, 0, sizeof(T0));
  for (int i = 0; i < (1 << (KT - 4)); ++i) T0.swz[i] = (uint8_t)hmap(uint32_t(i) << 4);
  for (int v = 0; v < 256; ++v)
    for (int j = 0; j < 8; ++j) {
      if (!(v >> j & 1)) continue;
      if (v < 64 && j < 6) T0.alo[v] += 1ull << slot[j];
      if (6 + j < KT) T0.ahi[v] += 1ull << slot[6 + j];
    }
  for (int v = 0; v < 64; ++v) T0.plo[v] = (uint16_t)v;
  for (int v = 0; v < 256; ++v) T0.phi[v] = (uint16_t)(v << 6);
  T = T0;
  std::memset(T.plo, 0, sizeof(T.plo));
  std::memset(T.phi, 0, sizeof(T.phi));
  for (int v = 0; v < 256; ++v)
    for (int k = 0; k < 8; ++k) {
      if (!(v >> k & 1)) continue;
      if (v < 64 && k < 6) T.plo[v] |= (uint16_t)(1u << sig_inv[k]);
      if (6 + k < KT) T.phi[v] |= (uint16_t)(1u << sig_inv[6 + k]);
    }
  // LDS: the tile (FP32) + step tables + tile tables statically, 8 KB per step
  const size_t static_lds =
      (size_t(1) << KT) * 8 + sizeof(PartBfStep) * kPartBfMaxSteps + (64 + (size_t(1) << (KT - 6))) * 10 +
      (size_t(1) << (KT - 4));
  // 13-qubit tiles: resident fragments (1024 threads) when the part's steps
  // fit LDS beside the tile, else streamed
  // (the three-piece split streams them at 13 qubits)
  const bool stream_u = KT >= 14 || (KT == 13 && (pieces == 3 || bf.part13 != 1 ||
                                                  (160 * 1024 - static_lds) / step_frag_bytes < size_t(ns)));
  const bool u_direct = KT == 13 && stream_u && bf.part13 == 2 && pieces == 2;
  const int max_steps = stream_u ? part_bf_max_steps(KT, pieces)
                                 : (int)std::min<size_t>(kPartBfMaxSteps, (160 * 1024 - static_lds) / step_frag_bytes);
  const size_t steps_off = 2 * sizeof(PartBfTables);
  const size_t own_off = part_tables_bytes(ns), bytes = own_off + frags.size() * 2;
  const size_t frag_off = P.checked ? P.frag_off : own_off;
  std::vector<unsigned char> host(bytes);
  std::memcpy(host.data(), &T0, sizeof(T0));
  std::memcpy(host.data() + sizeof(T0), &T, sizeof(T));
  std::memcpy(host.data() + steps_off, steps.data(), sizeof(PartBfStep) * ns);
  if (!frags.empty()) std::memcpy(host.data() + own_off, frags.data(), frags.size() * 2);
  if (int rc = ensure_scratch(scratch, bytes, stream, err)) return rc;
  if (hipMemcpyAsync(scratch->ptr, host.data(), bytes, hipMemcpyHostToDevice, stream) != hipSuccess) {
    *err = "fused upload failed";
    return HSV_ERR_DEVICE;
  }
  const uint64_t all = (n == 64) ? ~0ull : ((1ull << n) - 1);
  // tiles with a set bit in a slot outside live_slots hold only zeros (and
  // stay zero): they are skipped
  const uint64_t outer = all & ~tmask & live_slots;
  const uint64_t ntiles = 1ull << __builtin_popcountll(outer);
  if (tpw <= 0) tpw = stream_u ? 1 : 8;
  const int grid = (int)((ntiles + tpw - 1) / tpw);
  const uint64_t top = top_slots(outer, bf.tile_order);
  const auto* dev = static_cast<const unsigned char*>(scratch->ptr);
  const bool c128 = dtype == HSV_C128;
  int rc = HSV_OK;
  // more steps than fit in LDS at once: one pass per chunk of steps, the
  // last one with the layout change (a layout change alone: one pass, no steps)
  for (int s0 = 0; (s0 < ns || (ns == 0 && s0 == 0)) && rc == HSV_OK; s0 += std::max(max_steps, 1)) {
    const int cnt = std::min(max_steps, ns - s0);
    const size_t to = s0 + cnt >= ns ? sizeof(PartBfTables) : 0;
    const size_t so = steps_off + sizeof(PartBfStep) * s0;
    const size_t fo = frag_off + size_t(s0) * step_frag_bytes;
    if (KT == 12 && pieces == 3)
      c128 ? launch_part_bf<double, 12, false, false, 3>(amp, dev, to, so, fo, cnt, grid, stream, ntiles, outer, top, tpw, &rc)
           : launch_part_bf<float, 12, false, false, 3>(amp, dev, to, so, fo, cnt, grid, stream, ntiles, outer, top, tpw, &rc);
    else if (KT == 13 && pieces == 3)
      c128 ? launch_part_bf<double, 13, true, false, 3>(amp, dev, to, so, fo, cnt, grid, stream, ntiles, outer, top, tpw, &rc)
           : launch_part_bf<float, 13, true, false, 3>(amp, dev, to, so, fo, cnt, grid, stream, ntiles, outer, top, tpw, &rc);
    else if (KT == 12) c128 ? launch_part_bf<double, 12, false>(amp, dev, to, so, fo, cnt, grid, stream, ntiles, outer, top, tpw, &rc)
                       : launch_part_bf<float, 12, false>(amp, dev, to, so, fo, cnt, grid, stream, ntiles, outer, top, tpw, &rc);
    else if (KT == 13 && u_direct)
      c128 ? launch_part_bf<double, 13, true, true>(amp, dev, to, so, fo, cnt, grid, stream, ntiles, outer, top, tpw, &rc)
           : launch_part_bf<float, 13, true, true>(amp, dev, to, so, fo, cnt, grid, stream, ntiles, outer, top, tpw, &rc);
    else if (KT == 13 && stream_u)
      c128 ? launch_part_bf<double, 13, true>(amp, dev, to, so, fo, cnt, grid, stream, ntiles, outer, top, tpw, &rc)
           : launch_part_bf<float, 13, true>(amp, dev, to, so, fo, cnt, grid, stream, ntiles, outer, top, tpw, &rc);
    else if (KT == 13)
      c128 ? launch_part_bf<double, 13, false>(amp, dev, to, so, fo, cnt, grid, stream, ntiles, outer, top, tpw, &rc)
           : launch_part_bf<float, 13, false>(amp, dev, to, so, fo, cnt, grid, stream, ntiles, outer, top, tpw, &rc);
    else c128 ? launch_part_bf<double, 14, true>(amp, dev, to, so, fo, cnt, grid, stream, ntiles, outer, top, tpw, &rc)
              : launch_part_bf<float, 14, true>(amp, dev, to, so, fo, cnt, grid, stream, ntiles, outer, top, tpw, &rc);
  }
  if (rc) { *err = "wide bf16 fused kernel attribute setup failed"; return rc; }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    *err = std::string("fused launch: ") + hipGetErrorString(e);
    return HSV_ERR_DEVICE;
  }
  return HSV_OK;
}

// host: pinned memory for the device's answers: the part is prepared on the
// device, with the same steps and tables; null: on the host.
int part_apply_bf(void* amp, int n, int dtype, hipStream_t stream, DeviceScratch* scratch,
                  const std::vector<Lowered>& gates, uint64_t tile_qubits, const int* phys, const int* phys_after,
                  uint64_t live_slots, const BfTune& bf, std::string* err, int pieces, void* host = nullptr,
                  size_t host_bytes = 0) {
  std::vector<std::vector<std::vector<int>>> groups(1);
  if (host) {
    std::vector<std::vector<uint64_t>> masks(1);
    for (const Lowered& L : gates) {
      if (L.kind == K_IDENT) continue;
      uint64_t m = 0;
      for (int i = 0; i < L.nt + L.nc; ++i) {
        const int q = i < L.nt ? L.t[i] : L.c[i - L.nt];
        m |= 1ull << (phys ? phys[q] : q);
      }
      masks[0].push_back(m);
    }
    if (int rc = fused_plan_steps(stream, scratch, host, host_bytes, masks, 5, &groups, err)) return rc;
  }
  FusedPart P;
  if (int rc = part_prepare_bf(n, gates, tile_qubits, phys, phys_after, pieces, &groups[0], &P, err)) return rc;
  if (host)
    if (int rc = fused_parts_check(stream, scratch, host, host_bytes, &P, 1, pieces, err)) return rc;
  return part_launch_bf(amp, n, dtype, stream, scratch, P, live_slots, bf, pieces, err);
}

// The FP64 path on tiles (k_fused_tile). *taken = false, and nothing done, when
// the dense kernel is to run: a matrix that is not finite (a NaN spreads over
// the product that it is part of), a gate on more than 4 qubits, more steps than
// the dense product is worth (2^(K - 4) in FP64, which it has the same flops
// as; half as many again against the FP32-split product, whose three FP32
// products a flop take 1.5 times FP64's time), a state below a tile, or steps
// whose unitarity does not by itself bound the part's (a gate and its inverse
// that are not unitary, say): U^H U - I of a product of S embedded steps is at
// most 16 S times the steps' own in its largest entry.
int fused_apply_tile64(void* amp, int n, int dtype, hipStream_t stream, DeviceScratch* scratch,
                       const std::vector<Lowered>& gates, bool split, uint64_t live, int tile_order, bool* taken,
                       std::string* err) {
  *taken = false;
  std::vector<uint64_t> qm;
  std::vector<const Lowered*> gl;
  uint64_t pmask = 0;
  for (const Lowered& L : gates) {
    if (L.kind == K_IDENT) continue;
    if (!finite_matrix(L)) return HSV_OK;
    uint64_t m = 0;
    for (int i = 0; i < L.nt; ++i) m |= 1ull << L.t[i];
    for (int i = 0; i < L.nc; ++i) m |= 1ull << L.c[i];
    qm.push_back(m);
    gl.push_back(&L);
    pmask |= m;
  }
  const int K = std::max(4, __builtin_popcountll(pmask));
  // one workgroup per tile: its 2^(n - 12) * 512 threads must fit 32 bits
  if (n < 12 || n > 34 || K > 7 || qm.empty()) return HSV_OK;
  // the search ends where it exceeds what is worth it (120 gates on 7 qubits:
  // 0.2 of the 4.9 ms that preparing the dense product takes, 0.3 to its end)
  const int worth = std::min(kTileStepsMax, (split ? 3 : 2) << (K - 4) >> 1);
  const std::vector<std::vector<int>> groups = step_groups(qm, 4, 16, worth);
  const int ns = (int)groups.size();
  if (ns == 0) return HSV_OK;
  uint64_t tmask = pmask;
  for (int b = 0; b < n && __builtin_popcountll(tmask) < 12; ++b) tmask |= 1ull << b;
  int slot[12];
  for (int b = 0, j = 0; b < 64; ++b)
    if (tmask >> b & 1) slot[j++] = b;
  const size_t step_off = sizeof(TileAddr);
  const size_t frag_off = (step_off + sizeof(TileStep) * ns + 255) & ~size_t(255);
  std::vector<unsigned char> host(frag_off + size_t(ns) * 256 * sizeof(double2));
  auto* T = reinterpret_cast<TileAddr*>(host.data());
  for (int v = 0; v < 64; ++v)
    for (int j = 0; j < 6; ++j)
      if (v >> j & 1) {
        T->alo[v] += 1ull << slot[j];
        T->ahi[v] += 1ull << slot[6 + j];
      }
  auto* steps = reinterpret_cast<TileStep*>(host.data() + step_off);
  auto* frags = reinterpret_cast<double*>(host.data() + frag_off);
  for (int s = 0; s < ns; ++s) {
    uint64_t gm = 0;
    std::vector<Lowered> sg;
    for (int i : groups[s]) {
      gm |= qm[i];
      sg.push_back(*gl[i]);
    }
    for (int j = 0; j < 12 && __builtin_popcountll(gm) < 4; ++j) gm |= 1ull << slot[j];  // pad: U (x) I
    // columns: the four that index a quarter-wave's lanes first, with
    // distinct places modulo 4 where there are such (tile_sw moves tile bits
    // j, j + 4 and j + 8 onto the same LDS bank bit), then the others
    int rbit[4], cbit[8], nr = 0, nc = 0;
    std::vector<int> qubits, rest;
    bool used[4] = {false, false, false, false};
    for (int j = 0; j < 12; ++j) {
      if (gm >> slot[j] & 1) {
        rbit[nr++] = j;
        qubits.push_back(slot[j]);
      } else if (!used[j & 3]) {
        used[j & 3] = true;
        cbit[nc++] = j;
      } else {
        rest.push_back(j);
      }
    }
    for (int j : rest) cbit[nc++] = j;
    std::vector<cd> U;
    build_fused(sg, qubits, &U);
    if (!(16.0 * ns * unitarity_error(U, 16) <= 1e-10)) return HSV_OK;
    for (int v = 0; v < 16; ++v)
      for (int j = 0; j < 4; ++j)
        if (v >> j & 1) {
          steps[s].rt[v] ^= (uint16_t)tile_sw(1u << rbit[j]);
          steps[s].ctl[v] ^= (uint16_t)tile_sw(1u << cbit[j]);
          steps[s].cth[v] ^= (uint16_t)tile_sw(1u << cbit[4 + j]);
        }
    for (int ks = 0; ks < 4; ++ks)
      for (int lane = 0; lane < 64; ++lane) {
        const cd u = U[size_t(lane & 15) * 16 + 4 * ks + (lane >> 4)];
        double* f = frags + ((size_t(s) * 4 + ks) * 64 + lane) * 2;
        f[0] = u.real();
        f[1] = u.imag();
      }
  }
  *taken = true;
  if (int rc = ensure_scratch(scratch, host.size(), stream, err)) return rc;
  if (hipMemcpyAsync(scratch->ptr, host.data(), host.size(), hipMemcpyHostToDevice, stream) != hipSuccess) {
    *err = "fused upload failed";
    return HSV_ERR_DEVICE;
  }
  const uint64_t all = (n == 64) ? ~0ull : ((1ull << n) - 1);
  const uint64_t outer = all & ~tmask & live, top = top_slots(outer, tile_order);
  const unsigned ntiles = 1u << __builtin_popcountll(outer);
  const auto* dev = static_cast<const unsigned char*>(scratch->ptr);
  const auto* da = reinterpret_cast<const TileAddr*>(dev);
  const auto* ds = reinterpret_cast<const TileStep*>(dev + step_off);
  const auto* df = reinterpret_cast<const double2*>(dev + frag_off);
  if (dtype == HSV_C128)
    hipLaunchKernelGGL((k_fused_tile<double>), ntiles, kTileThreads, 0, stream, static_cast<double2*>(amp), da, ds, df,
                       ns, outer, top);
  else
    hipLaunchKernelGGL((k_fused_tile<float>), ntiles, kTileThreads, 0, stream, static_cast<float2*>(amp), da, ds, df,
                       ns, outer, top);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    *err = std::string("fused launch: ") + hipGetErrorString(e);
    return HSV_ERR_DEVICE;
  }
  return HSV_OK;
}

// variant: 0 / 1 = column-block kernel (1: swizzled row order), 2 = tile form
// (needs n >= 12; falls back to 1 below that).
int fused_apply_bf(void* amp, int n, int dtype, hipStream_t stream, int num_cu, DeviceScratch* scratch,
                   const std::vector<int>& Q, const std::vector<cd>& Um, uint64_t live, int variant, int tpw,
                   int tile_order, std::string* err) {
  const int K = (int)Q.size();
  const int D = 1 << K;
  if (K < 5 || K > 7) {
    *err = "the bf16 fused path takes parts of 5..7 qubits";
    return HSV_ERR_LIMIT;
  }
  const bool tile = variant == 2 && n >= 12;
  const int swizzle = variant >= 1 ? 1 : 0;
  const int RB = D / 16, KS = D / 32;
  const size_t frag_bytes = size_t(8) * D * D;
  std::vector<unsigned char> host(frag_bytes + std::max(size_t(D) * 8 + 16 * 8, sizeof(BfTileTables)));
  uint16_t* hf = reinterpret_cast<uint16_t*>(host.data());
  for (int rb = 0; rb < RB; ++rb)
    for (int ks = 0; ks < KS; ++ks)
      for (int lane = 0; lane < 64; ++lane)
        for (int e = 0; e < 8; ++e) {
          const int mm = lane % 16, g = lane / 16;
          const int row = 16 * rb + (swizzle ? 4 * (mm % 4) + mm / 4 : mm);
          const int col = 32 * ks + (swizzle ? g + 4 * e : 8 * g + e);
          const cd u = Um[size_t(row) * D + col];
          const uint16_t rh = bf16_bits((float)u.real()), ih = bf16_bits((float)u.imag());
          const uint16_t rl = bf16_bits((float)(u.real() - bf16_value(rh)));
          const uint16_t il = bf16_bits((float)(u.imag() - bf16_value(ih)));
          const size_t frag = size_t((rb * KS + ks) * 4) * 64;  // first of the 4 sets, in 8-element units
          hf[(frag + 0 * 64 + lane) * 8 + e] = rh;
          hf[(frag + 1 * 64 + lane) * 8 + e] = rl;
          hf[(frag + 2 * 64 + lane) * 8 + e] = ih;
          hf[(frag + 3 * 64 + lane) * 8 + e] = il;
        }
  uint64_t qmask = 0;
  for (int q : Q) qmask |= 1ull << q;
  const uint64_t all = (n == 64) ? ~0ull : ((1ull << n) - 1);
  if (tile) {
    uint64_t cmask = 0;
    for (int b = 0, got = 0; b < n && got < 12 - K; ++b)
      if (!(qmask >> b & 1)) { cmask |= 1ull << b; ++got; }
    build_tile_tables(qmask, cmask, reinterpret_cast<BfTileTables*>(host.data() + frag_bytes));
    const size_t bytes = frag_bytes + sizeof(BfTileTables);
    if (int rc = ensure_scratch(scratch, bytes, stream, err)) return rc;
    if (hipMemcpyAsync(scratch->ptr, host.data(), bytes, hipMemcpyHostToDevice, stream) != hipSuccess) {
      *err = "fused upload failed";
      return HSV_ERR_DEVICE;
    }
    const uint64_t outer = all & ~qmask & ~cmask & live;
    const uint64_t ntiles = 1ull << __builtin_popcountll(outer);
    const int grid = (int)((ntiles + tpw - 1) / tpw);
    const uint64_t top = top_slots(outer, tile_order);
    const bool c128 = dtype == HSV_C128;
    if (K == 5) c128 ? launch_bft<double, 5>(amp, scratch->ptr, grid, stream, ntiles, outer, top, tpw)
                     : launch_bft<float, 5>(amp, scratch->ptr, grid, stream, ntiles, outer, top, tpw);
    else if (K == 6) c128 ? launch_bft<double, 6>(amp, scratch->ptr, grid, stream, ntiles, outer, top, tpw)
                          : launch_bft<float, 6>(amp, scratch->ptr, grid, stream, ntiles, outer, top, tpw);
    else c128 ? launch_bft<double, 7>(amp, scratch->ptr, grid, stream, ntiles, outer, top, tpw)
              : launch_bft<float, 7>(amp, scratch->ptr, grid, stream, ntiles, outer, top, tpw);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
      *err = std::string("fused launch: ") + hipGetErrorString(e);
      return HSV_ERR_DEVICE;
    }
    return HSV_OK;
  }
  uint64_t tmask = 0;
  for (int b = 0, got = 0; b < n && got < 4; ++b)
    if (!(qmask >> b & 1)) { tmask |= 1ull << b; ++got; }
  uint64_t* hq = reinterpret_cast<uint64_t*>(host.data() + frag_bytes);
  for (int r = 0; r < D; ++r) hq[r] = pdep_host((uint64_t)r, qmask);
  for (int c = 0; c < 16; ++c) hq[D + c] = pdep_host((uint64_t)c, tmask);
  const size_t bytes = frag_bytes + size_t(D) * 8 + 16 * 8;
  if (int rc = ensure_scratch(scratch, bytes, stream, err)) return rc;
  if (hipMemcpyAsync(scratch->ptr, host.data(), bytes, hipMemcpyHostToDevice, stream) != hipSuccess) {
    *err = "fused upload failed";
    return HSV_ERR_DEVICE;
  }
  BfArgs f{};
  f.outer_mask = all & ~qmask & ~tmask & live;
  f.nblocks = 1ull << __builtin_popcountll(f.outer_mask);
  const uint64_t waves = kBfThreads / 64;
  const int grid = (int)std::min<uint64_t>((f.nblocks + waves - 1) / waves, uint64_t(num_cu) * 2);
  int rc = HSV_OK;
  const bool c128 = dtype == HSV_C128;
#define HSV_BF_LAUNCH(K_, S_)                                                                  \
  (c128 ? launch_bf<double, K_, S_>(amp, scratch->ptr, grid, stream, f, &rc)                  \
        : launch_bf<float, K_, S_>(amp, scratch->ptr, grid, stream, f, &rc))
  if (swizzle) {
    if (K == 5) HSV_BF_LAUNCH(5, true); else if (K == 6) HSV_BF_LAUNCH(6, true); else HSV_BF_LAUNCH(7, true);
  } else {
    if (K == 5) HSV_BF_LAUNCH(5, false); else if (K == 6) HSV_BF_LAUNCH(6, false); else HSV_BF_LAUNCH(7, false);
  }
#undef HSV_BF_LAUNCH
  if (rc) { *err = "bf16 fused kernel attribute setup failed"; return rc; }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    *err = std::string("fused launch: ") + hipGetErrorString(e);
    return HSV_ERR_DEVICE;
  }
  return HSV_OK;
}

}  // namespace

int fused_part_prepare(int n, const std::vector<Lowered>& gates, uint64_t tile_qubits, const int* phys,
                       const int* phys_after, int pieces, const std::vector<std::vector<int>>* groups, FusedPart* part,
                       std::string* err) {
  return part_prepare_bf(n, gates, tile_qubits, phys, phys_after, pieces, groups, part, err);
}

int fused_part_launch(void* amp, int n, int dtype, hipStream_t stream, DeviceScratch* scratch, const FusedPart& part,
                      uint64_t live_slots, const BfTune& bf, int pieces, std::string* err) {
  return part_launch_bf(amp, n, dtype, stream, scratch, part, live_slots, bf, pieces, err);
}

int fused_part_bf_layout(void* amp, int n, int dtype, hipStream_t stream, DeviceScratch* scratch,
                         const std::vector<Lowered>& gates, uint64_t tile_qubits, const int* phys,
                         const int* phys_after, uint64_t live_slots, const BfTune& bf, std::string* err,
                         int pieces) {
  return part_apply_bf(amp, n, dtype, stream, scratch, gates, tile_qubits, phys, phys_after, live_slots, bf, err,
                       pieces);
}

int fused_parts_check(hipStream_t stream, DeviceScratch* scratch, void* host, size_t host_bytes, FusedPart* parts,
                      int count, int pieces, std::string* err) {
  // the answers in host: 14 swizzle images a part, then an error a step
  std::vector<SwizzlePart> sw;
  std::vector<PartSwizzleKey> keys;
  std::vector<cd> U;
  std::vector<int> which;
  size_t ns = 0, tables = 0;
  for (int p = 0; p < count; ++p) {
    const FusedPart& P = parts[p];
    if (P.steps.empty()) continue;
    if ((sw.size() + 1) * 14 * sizeof(uint32_t) + 8 + (ns + P.steps.size()) * sizeof(double) > host_bytes) break;
    int sig_inv[14];
    const std::vector<PartSwizzleKey> k = part_keys(P, sig_inv);
    sw.push_back(SwizzlePart{P.KT, (int)keys.size(), (int)k.size()});
    keys.insert(keys.end(), k.begin(), k.end());
    for (const FusedPart::Step& S : P.steps) U.insert(U.end(), S.U.begin(), S.U.end());
    which.push_back(p);
    ns += P.steps.size();
    tables = std::max(tables, part_tables_bytes(P.steps.size()));
  }
  // parts without steps (a layout change alone) have tables too
  tables = std::max(tables, part_tables_bytes(0));
  if (which.empty()) return HSV_OK;
  std::vector<uint64_t> rng(kSwizzleThreads);
  uint64_t r = kSwizzleSeed;
  uint32_t cand[14];
  for (size_t t = 0; t < rng.size(); ++t) {
    rng[t] = r;
    for (int e = 0; e < kSwizzleEach; ++e) swizzle_candidate(&r, 14, cand);
  }
  // scratch: tables of the part under way | fragments | matrices | generator
  // states | parts | keys
  const size_t step_frag = size_t(2) * 2 * pieces * 64 * 16, u_off = tables + ns * step_frag,
               rng_off = u_off + U.size() * sizeof(cd), sw_off = rng_off + rng.size() * sizeof(uint64_t),
               key_off = sw_off + sw.size() * sizeof(SwizzlePart), end = key_off + keys.size() * sizeof(PartSwizzleKey);
  std::vector<unsigned char> up(end - u_off);
  std::memcpy(up.data(), U.data(), U.size() * sizeof(cd));
  std::memcpy(up.data() + (rng_off - u_off), rng.data(), rng.size() * sizeof(uint64_t));
  std::memcpy(up.data() + (sw_off - u_off), sw.data(), sw.size() * sizeof(SwizzlePart));
  std::memcpy(up.data() + (key_off - u_off), keys.data(), keys.size() * sizeof(PartSwizzleKey));
  if (int rc = ensure_scratch(scratch, end, stream, err)) {
    if (rc != HSV_ERR_ALLOC) return rc;
    (void)hipGetLastError();  // no room on the card: the host's way
    err->clear();
    return HSV_OK;
  }
  auto* dev = static_cast<unsigned char*>(scratch->ptr);
  auto* nimg = static_cast<uint32_t*>(host);
  auto* uerr = reinterpret_cast<double*>(static_cast<unsigned char*>(host) +
                                         ((sw.size() * 14 * sizeof(uint32_t) + 7) & ~size_t(7)));
  if (hipMemcpyAsync(dev + u_off, up.data(), up.size(), hipMemcpyHostToDevice, stream) != hipSuccess) {
    *err = "fused upload failed";
    return HSV_ERR_DEVICE;
  }
  hipLaunchKernelGGL(k_part_steps, (unsigned)ns, kStepThreads, 0, stream, reinterpret_cast<const double2*>(dev + u_off),
                     pieces, reinterpret_cast<uint16_t*>(dev + tables), uerr);
  hipLaunchKernelGGL(k_part_swizzle, (unsigned)sw.size(), kSwizzleThreads, 0, stream,
                     reinterpret_cast<const SwizzlePart*>(dev + sw_off),
                     reinterpret_cast<const PartSwizzleKey*>(dev + key_off),
                     reinterpret_cast<const uint64_t*>(dev + rng_off), nimg);
  if (hipGetLastError() != hipSuccess || hipStreamSynchronize(stream) != hipSuccess) {
    *err = "the step check failed on the device";
    return HSV_ERR_DEVICE;
  }
  size_t s0 = 0;
  for (size_t w = 0; w < which.size(); ++w) {
    FusedPart& P = parts[which[w]];
    P.checked = true;
    P.uerr.assign(uerr + s0, uerr + s0 + P.steps.size());
    std::memcpy(P.nimg, nimg + w * 14, sizeof(P.nimg));
    P.frag_off = tables + s0 * step_frag;
    s0 += P.steps.size();
  }
  return HSV_OK;
}

int fused_plan_steps(hipStream_t stream, DeviceScratch* scratch, void* host, size_t host_bytes,
                     const std::vector<std::vector<uint64_t>>& masks, int k,
                     std::vector<std::vector<std::vector<int>>>* groups, std::string* err) {
  groups->assign(masks.size(), {});
  struct Wanted {
    size_t part;
    uint64_t all;
    std::vector<int> live;  // its gates that act on something
  };
  auto* base = static_cast<unsigned char*>(host);
  size_t p0 = 0;
  while (p0 < masks.size()) {
    // as many parts as the buffer takes: headers | gate masks | answers
    std::vector<Wanted> want;
    size_t gates = 0;
    double work = 0;
    for (; p0 < masks.size(); ++p0) {
      Wanted w{p0, 0, {}};
      bool fits = true;
      for (size_t i = 0; i < masks[p0].size(); ++i) {
        if (!masks[p0][i]) continue;
        w.live.push_back((int)i);
        w.all |= masks[p0][i];
        fits = fits && __builtin_popcountll(masks[p0][i]) <= k;
      }
      const int nq = __builtin_popcountll(w.all);
      if (!fits || w.live.size() < 2 || w.live.size() > size_t(kPlanGates) || nq > kPlanQubits ||
          binomial(nq, std::min(k, nq)) > kPlanSubsets)
        continue;
      const size_t need = (want.size() + 1) * sizeof(PlanPart) + (gates + w.live.size()) * 4 + (want.size() + 1) * 2;
      if (need > host_bytes || want.size() == kPlanParts) break;
      gates += w.live.size();
      work += double(binomial(nq, std::min(k, nq))) * double(w.live.size());
      want.push_back(std::move(w));
    }
    // the host's search takes about 40 ns a subset and gate, the device's
    // (launch and wait included) about 0.5 to 1 ms whatever the number of parts
    if (want.empty() || work < kPlanWork) continue;
    auto* parts = reinterpret_cast<PlanPart*>(base);
    auto* gm = reinterpret_cast<uint16_t*>(base + want.size() * sizeof(PlanPart));
    auto* out = gm + gates;
    int mo = 0, oo = 0;
    for (size_t w = 0; w < want.size(); ++w) {
      parts[w] = PlanPart{(int)want[w].live.size(), __builtin_popcountll(want[w].all), mo, oo};
      for (int i : want[w].live) {
        // qubit bits to the part's own, ascending
        uint32_t c = 0;
        int j = 0;
        for (uint64_t a = want[w].all; a; a &= a - 1, ++j)
          if (masks[want[w].part][i] & a & (~a + 1)) c |= 1u << j;
        gm[mo++] = (uint16_t)c;
      }
      oo += (int)want[w].live.size() + 1;
    }
    if (int rc = ensure_scratch(scratch, want.size() * sizeof(PlanState), stream, err)) {
      if (rc != HSV_ERR_ALLOC) return rc;
      (void)hipGetLastError();  // no room on the card: the rest is searched on the host
      err->clear();
      return HSV_OK;
    }
    auto* st = static_cast<PlanState*>(scratch->ptr);
    const unsigned np = (unsigned)want.size();
    size_t most = 0;
    int blocks = 0;
    for (size_t w = 0; w < want.size(); ++w) {
      most = std::max(most, want[w].live.size());
      const int nq = parts[w].num_qubits;
      blocks = std::max(blocks, (binomial(nq, std::min(k, nq)) + kPlanThreads - 1) / kPlanThreads);
    }
    hipLaunchKernelGGL(k_plan_start, np, kPlanThreads, 0, stream, parts, gm, k, st, out);
    for (int level = 0; level < std::min<int>(kPlanLevels, (int)most); ++level) {
      hipLaunchKernelGGL(k_plan_score, dim3(blocks, np, level ? kPlanWidth : 1), kPlanThreads, 0, stream, parts, k,
                         level, st);
      hipLaunchKernelGGL(k_plan_select, np, kPlanSelect, 0, stream, parts, k, level, st, out);
    }
    if (hipGetLastError() != hipSuccess || hipStreamSynchronize(stream) != hipSuccess) {
      *err = "step grouping failed on the device";
      return HSV_ERR_DEVICE;
    }
    for (size_t w = 0; w < want.size(); ++w) {
      const uint16_t* o = out + parts[w].out;
      const uint16_t* m = gm + parts[w].masks;
      // the sets' blocking scans, one after another (none when not found)
      std::vector<int> rem(want[w].live.size());
      for (size_t i = 0; i < rem.size(); ++i) rem[i] = (int)i;
      for (int g = 0; g < o[0]; ++g) {
        const uint32_t Q = o[1 + g];
        uint32_t blocked = 0;
        std::vector<int> taken, keep;
        for (int i : rem) {
          if ((m[i] & blocked) || (m[i] & ~Q)) {
            blocked |= m[i];
            keep.push_back(i);
          } else {
            taken.push_back(want[w].live[i]);
          }
        }
        (*groups)[want[w].part].push_back(std::move(taken));
        rem.swap(keep);
      }
      if (!rem.empty()) (*groups)[want[w].part].clear();
    }
  }
  return HSV_OK;
}

int fused_apply(void* amp, int n, int dtype, hipStream_t stream, int num_cu, DeviceScratch* scratch,
                const std::vector<Lowered>& gates, int mode, uint64_t live, std::string* err, const BfTune& bf,
                void* pinned, size_t pinned_bytes) {
  if (mode != HSV_FUSED_F64 && mode != HSV_FUSED_F32SPLIT && mode != HSV_FUSED_BF16SPLIT &&
      mode != HSV_FUSED_BF16X3) {
    *err = "unknown fused mode";
    return HSV_ERR_ARG;
  }
  if (mode == HSV_FUSED_BF16X3) {
    // the three-piece split runs every part on the wide-part kernel, in a
    // 12- or 13-qubit tile with slots 0-4
    uint64_t pmask = 0;
    for (const Lowered& L : gates) {
      if (L.kind == K_IDENT) continue;
      for (int i = 0; i < L.nt; ++i) pmask |= 1ull << L.t[i];
      for (int i = 0; i < L.nc; ++i) pmask |= 1ull << L.c[i];
    }
    return part_apply_bf(amp, n, dtype, stream, scratch, gates, pmask, nullptr, nullptr, live, bf, err, 3, pinned,
                         pinned_bytes);
  }
  if (mode == HSV_FUSED_BF16SPLIT) {
    uint64_t pmask = 0;
    for (const Lowered& L : gates) {
      if (L.kind == K_IDENT) continue;
      for (int i = 0; i < L.nt; ++i) pmask |= 1ull << L.t[i];
      for (int i = 0; i < L.nc; ++i) pmask |= 1ull << L.c[i];
    }
    if (__builtin_popcountll(pmask) > 7)
      return part_apply_bf(amp, n, dtype, stream, scratch, gates, pmask, nullptr, nullptr, live, bf, err, 2, pinned,
                           pinned_bytes);
  }
  if (mode == HSV_FUSED_F64 || mode == HSV_FUSED_F32SPLIT) {
    // identities count towards a part's 7 qubits
    uint64_t mask = 0;
    for (const Lowered& L : gates) {
      for (int i = 0; i < L.nt; ++i) mask |= 1ull << L.t[i];
      for (int i = 0; i < L.nc; ++i) mask |= 1ull << L.c[i];
    }
    bool taken = false;
    if (__builtin_popcountll(mask) <= 7)
      if (int rc = fused_apply_tile64(amp, n, dtype, stream, scratch, gates, mode == HSV_FUSED_F32SPLIT, live, bf.tile_order, &taken, err)) return rc;
    if (taken) return HSV_OK;
  }
  std::vector<int> Q;
  std::vector<cd> Um;
  if (int rc = fused_unitary(n, gates, &Q, &Um, err, mode == HSV_FUSED_BF16SPLIT ? 5 : 4)) return rc;
  const int K = (int)Q.size();
  const int D = 1 << K;
  const double uerr = unitarity_error(Um, D);
  if (!(uerr <= 1e-10)) {
    *err = "fused matrix is not unitary (max |U^H U - I| = " + std::to_string(uerr) + ")";
    return HSV_ERR_UNITARY;
  }
  const int free_bits = n - K;
  if (free_bits < 4) {
    *err = "fused parts need at least 4 state qubits outside the part";
    return HSV_ERR_LIMIT;
  }
  if (mode == HSV_FUSED_BF16SPLIT)
    return fused_apply_bf(amp, n, dtype, stream, num_cu, scratch, Q, Um, live, bf.variant, std::max(bf.tile_tpw, 1),
                          bf.tile_order, err);
  int NC = 2048 / (16 * D);
  while (NC > 1 && 4 + __builtin_ctz(NC) > free_bits) NC >>= 1;
  const int C = 16 * NC;
  const int logC = __builtin_ctz(C);
  uint64_t qmask = 0;
  for (int q : Q) qmask |= 1ull << q;
  uint64_t tmask = 0;
  for (int b = 0, got = 0; b < n && got < logC; ++b)
    if (!(qmask >> b & 1)) { tmask |= 1ull << b; ++got; }
  const uint64_t all = (n == 64) ? ~0ull : ((1ull << n) - 1);
  FusedArgs f{};
  f.outer_mask = all & ~qmask & ~tmask & live;
  f.ntiles = 1ull << __builtin_popcountll(f.outer_mask);
  f.C = C;
  f.logC = logC;
  f.NC = NC;
  // scratch layout: U (D*D double2) | qoff (D u64) | toff (C u64)
  std::vector<unsigned char> host(size_t(D) * D * 16 + size_t(D) * 8 + size_t(C) * 8);
  double* hu = reinterpret_cast<double*>(host.data());
  for (size_t i = 0; i < size_t(D) * D; ++i) { hu[2 * i] = Um[i].real(); hu[2 * i + 1] = Um[i].imag(); }
  uint64_t* hq = reinterpret_cast<uint64_t*>(host.data() + size_t(D) * D * 16);
  for (int r = 0; r < D; ++r) hq[r] = pdep_host((uint64_t)r, qmask);
  uint64_t* ht = hq + D;
  for (int c = 0; c < C; ++c) ht[c] = pdep_host((uint64_t)c, tmask);
  if (int rc = ensure_scratch(scratch, host.size(), stream, err)) return rc;
  if (hipMemcpyAsync(scratch->ptr, host.data(), host.size(), hipMemcpyHostToDevice, stream) != hipSuccess) {
    *err = "fused upload failed";
    return HSV_ERR_DEVICE;
  }
  const int per_cu = K >= 7 ? 2 : 4;
  const int grid = (int)std::min<uint64_t>(f.ntiles, uint64_t(num_cu) * per_cu);
  const bool split = mode == HSV_FUSED_F32SPLIT;
  if (dtype == HSV_C128) {
    if (split) launch_k<double, true>(K, amp, scratch->ptr, D, C, grid, stream, f);
    else launch_k<double, false>(K, amp, scratch->ptr, D, C, grid, stream, f);
  } else {
    if (split) launch_k<float, true>(K, amp, scratch->ptr, D, C, grid, stream, f);
    else launch_k<float, false>(K, amp, scratch->ptr, D, C, grid, stream, f);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    *err = std::string("fused launch: ") + hipGetErrorString(e);
    return HSV_ERR_DEVICE;
  }
  return HSV_OK;
}

}  // namespace hsv
