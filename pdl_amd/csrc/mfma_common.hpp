// What the split-FP16 and FP8 kernels of k_mfma.hip and the split-FP16
// product of k_hgemm.hip share: operand types, the finishing of an output,
// the packed panels' layout and the order of tiles.
#pragma once

#include <hip/hip_runtime.h>

#include "device.hpp"

namespace pdlhip {

typedef _Float16 half_t;
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// exponent of a power of two held as a normal float
__device__ __forceinline__ int pow2_exp(float s) { return ((__float_as_int(s) >> 23) & 0xff) - 127; }

// Whether output c (unscaled; the accumulator was c * 2^e) must come from
// PDL's loop: the range-loss bound (D_A[h] + D_B[w]) * 2^15 (scaled units)
// exceeds 2^-22 |c|, or c is not finite.  The GEMM epilogue and the fixup
// kernel evaluate the same test on the same stored c.
__device__ __forceinline__ bool mm_needs_fix(float c, float dd, int e) {
  if (dd == 0.0f && fabsf(c) < __builtin_inff()) return false;
  return !(ldexpf(dd * 32768.0f, -e) <= 0x1p-22f * fabsf(c));
}

// the GEMM epilogue for one output: unscale the accumulator exactly and
// mark the row of an output the fixup kernel must recompute
__device__ __forceinline__ float mm_finish(float v, float da, float db, float sa, float sb, int *rowflag, int64_t h) {
  const int e = pow2_exp(sa) + pow2_exp(sb);
  const float c = ldexpf(v, -e);
  if (mm_needs_fix(c, da + db, e)) rowflag[h] = 1;   // the same value from every writer
  return c;
}

// Packed FP16 panels of an operand of R rows x K (both padded): pieces of 32
// rows x 16 k in the order [row / 32][k / 16][hi, lo], each 1 KiB and laid out
// as it lies in LDS, so that one wave moves a piece with one load of 16 bytes
// per lane from 1 KiB of consecutive memory.  Within a piece a row's two
// 16-byte halves change places with bit 2 of the row: eight rows' reads of
// one half then fall on distinct LDS banks.
constexpr int PIECE = 32 * 16;   // halves
// element offset of the 8 k of `row` that start at k (a multiple of 8) in the hi piece; lo is PIECE further on
__host__ __device__ __forceinline__ int64_t panel_at(int64_t row, int64_t k, int64_t Kp) {
  const int rr = (int)(row & 31), half = (int)(k >> 3) & 1;
  return ((row >> 5) * (Kp >> 4) + (k >> 4)) * (2 * PIECE) + rr * 16 + ((half ^ (rr >> 2 & 1)) * 8);
}

// block -> C tile.  The 8 XCDs take blocks round-robin (block b runs on XCD
// b % 8), so each XCD is given one contiguous share of the tile order; within
// a share, tiles go in groups of 8 tile-rows, column by column, so the blocks
// resident on one XCD at a time reuse the same A row-panels and B
// column-panels from that XCD's L2.
__device__ inline void tile_of(int64_t b, int64_t ntm, int64_t ntn, int64_t &tm, int64_t &tn) {
  const int64_t nb = ntm * ntn;
  const int64_t t = (nb % 8 == 0) ? (b % 8) * (nb / 8) + b / 8 : b;
  constexpr int64_t G = 8;
  const int64_t g = t / (G * ntn), r = t % (G * ntn);
  const int64_t rows = ntm - g * G < G ? ntm - g * G : G;
  tm = g * G + r % rows;
  tn = r / rows;
}

// one wave's direct global -> LDS load: lane i's 16 bytes go to l + 16 * i
template <class T> __device__ __forceinline__ void dma16(const T *g, T *l) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)g,
                                   (__attribute__((address_space(3))) void *)l, 16, 0, 0);
}

// C tile products of packed panels (k_hgemm.hip): blocks of 256x256 or 128x128
hipError_t launch_split16(bool big, const half_t *A, const half_t *B, const float *sA, const float *sB, const float *dA,
                          const float *dB, int *rowflag, float *c, const MmPlan &p, int64_t Kp, int64_t ntm, int64_t ntn,
                          hipStream_t s);

}  // namespace pdlhip
