// Float and double matmult on the FP32 / FP64 matrix cores in the default
// precision mode (lib/PDL/Primitive.pd:191-245: C[h][w] = sum_t A[h][t]
// B[t][w]), single products and batches: the tiles of mm_tile.hpp.
//
// Bound by the matrix cores (32 or 64 cycles per instruction), so the tiles
// are small: 64x64 of C per block of 4 waves keeps four blocks resident per
// CU, whose waves cover each other's loads and barriers, and cuts a product
// into enough blocks for 256 CUs.  Double: 4096^3 2.09 ms, 65.8 TFLOP/s
// (128x128 blocks of the same kernel 2.33 ms, 128x64 2.28); 1500^3 132 + 4 us
// for the join in a trace, 119 a call among others (before, 144 blocks of
// 128x128: 277); 512^3 18 us (the SIMT kernel: 85).  One stage of loads in flight
// instead of two: 59 instead of 54 us at 1024^3, where a CU has one block.
// Float: 1024^3 30 us (packed for the FP16 split 70), 300^3 12 (46), 1413 x
// 1452 x 19 16 (the SIMT kernel 184), 128 x 8192 x 128 23 (174), 65536 of 32^3
// 0.17 ms (0.50).  Float tiles with a total and a partial sum per output (see
// mm_tile.hpp) take three blocks per CU: kept to the 128 registers of four,
// their loop spills and waits for its loads (1024^3: 36 us).
//
// Tiles that would fill only part of the chip in the last wave of blocks are
// cut along t into S parts, each summed into scratch, and joined by a second
// small kernel in a fixed order.
#include <hip/hip_runtime.h>

#include <type_traits>
#include <vector>

#include "device.hpp"
#include "launch.hpp"
#include "mm_tile.hpp"

namespace pdlhip {

void *partials_alloc(size_t bytes);
void partials_free(void *p);
bool small_split16(const MmPlan &p);    // k_mfma.hip: what the FP16 split's batch kernel takes
bool single_split16(const MmPlan &p);   // and its large product

template <class T> struct TilePlan {
  MmPlan p;
  int64_t ntm, ntn;    // tiles of one product
  int64_t nwhole;      // tiles summed over all of t; the others in S parts of kc
  int32_t S;
  int64_t kc;
  T *part;
};

// tile t of all products -> product, tile row, tile column: groups of 8 tile
// rows column by column, for the L2's sake
template <class T>
__device__ inline void tile_at(const TilePlan<T> &g, int64_t t, int64_t *o, int64_t &tm, int64_t &tn) {
  const int64_t per = g.ntm * g.ntn;
  int64_t bidx = per == 1 ? t : t / per;
  t -= bidx * per;
  constexpr int64_t G = 8;
  const int64_t q = t / (G * g.ntn), r = t % (G * g.ntn);
  const int64_t rows = g.ntm - q * G < G ? g.ntm - q * G : G;
  tm = q * G + r % rows;
  tn = r / rows;
  o[0] = g.p.off[0]; o[1] = g.p.off[1]; o[2] = g.p.off[2];
  for (int d = 0; d < g.p.nd; d++) {
    const int64_t i = d == g.p.nd - 1 ? bidx : bidx % g.p.dims[d];
    if (d < g.p.nd - 1) bidx /= g.p.dims[d];
    o[0] += i * g.p.inc[0][d]; o[1] += i * g.p.inc[1][d]; o[2] += i * g.p.inc[2][d];
  }
}

template <class T, int BM, int BN, int WR, int WC, bool AK, bool BK, int HOW>
__global__ __launch_bounds__(256, sizeof(T) == 4 && HOW == BY_STAGE ? 3 : 4) void tile_gemm(const T *__restrict__ a, const T *__restrict__ b, T *__restrict__ c,
                                                    TilePlan<T> g) {
  __shared__ __align__(16) T sA[TILE_BUFS<HOW>][BM][TILE_P<T>];
  __shared__ __align__(16) T sB[TILE_BUFS<HOW>][BN][TILE_P<T>];
  const MmPlan &p = g.p;
  // whole tiles first, each XCD (block b runs on XCD b % 8) a contiguous
  // share of them, then the parts
  int64_t t = blockIdx.x, kb = 0, ke = p.T;
  int part = -1;
  if (t < g.nwhole) {
    if (g.nwhole % 8 == 0) t = (t % 8) * (g.nwhole / 8) + t / 8;
  } else {
    const int64_t r = t - g.nwhole;
    part = (int)(r % g.S);
    t = g.nwhole + r / g.S;
    kb = part * g.kc;
    ke = kb + g.kc < p.T ? kb + g.kc : p.T;
  }
  int64_t o[3], tm, tn;
  tile_at(g, t, o, tm, tn);
  const int64_t m0 = tm * BM, n0 = tn * BN;
  T *dst = part >= 0 ? g.part + ((t - g.nwhole) * g.S + part) * (BM * BN) : c + o[2] + n0 * p.c_w + m0 * p.c_h;
  const int64_t dh = part >= 0 ? BN : p.c_h, dw = part >= 0 ? 1 : p.c_w;
  const int64_t rows = part >= 0 ? BM : p.H - m0, cols = part >= 0 ? BN : p.W - n0;
  tile_product<T, BM, BN, WR, WC, AK, BK, HOW>(a + o[0], b + o[1], p.H, p.W, p.a_h, p.a_t, p.b_w, p.b_t, m0, n0, kb, ke, sA,
                                          sB, [&](int h, int w, T v) {
                                            if (h < rows && w < cols) dst[h * dh + w * dw] = v;
                                          });
}

// the parts of each cut tile, added in ascending t
template <class T, int BM, int BN>
__global__ __launch_bounds__(256) void tile_join(T *__restrict__ c, TilePlan<T> g) {
  constexpr int PER = BM * BN / 256;
  const int64_t q = blockIdx.x / PER;
  const int e = (int)(blockIdx.x % PER) * 256 + threadIdx.x, h = e / BN, wv = e % BN;
  const T *src = g.part + q * g.S * (BM * BN) + e;
  T s = src[0];
  for (int k = 1; k < g.S; k++) s += src[(int64_t)k * (BM * BN)];
  int64_t o[3], tm, tn;
  tile_at(g, g.nwhole + q, o, tm, tn);
  if (tm * BM + h < g.p.H && tn * BN + wv < g.p.W)
    c[o[2] + (tn * BN + wv) * g.p.c_w + (tm * BM + h) * g.p.c_h] = s;
}

// Into how many parts the tiles past the last multiple of 256 (a tile per CU)
// are cut: whole, they leave CUs idle for a whole tile's time.  S parts make
// that ceil(rest * S / 256) / S of it, for a second launch and the parts'
// traffic (about 4 us); a part keeps at least 64 k.
template <class T> static int tile_parts(int64_t rest, int BM, int BN, int64_t K) {
  constexpr double CU_FLOPS = sizeof(T) == 8 ? 0.24e6 : 0.44e6;   // per us and CU, as measured
  const double tile_us = 2.0 * BM * BN * (double)K / CU_FLOPS;
  int parts = 1;
  double best = rest ? tile_us : 0.0;
  for (int S = 2; S <= 16 && rest && K / S >= 64; S++) {
    const double us = tile_us * (double)((rest * S + 255) / 256) / S + 4.0 + (double)(rest * S * BM * BN * 2 * sizeof(T)) / 3e6;
    if (us < best) { best = us; parts = S; }
  }
  return parts;
}

template <class T, int BM, int BN, int WR, int WC>
static hipError_t tile_launch(const MmPlan &p, const T *a, const T *b, T *c, hipStream_t s) {
  TilePlan<T> g;
  g.p = p;
  g.ntm = (p.H + BM - 1) / BM;
  g.ntn = (p.W + BN - 1) / BN;
  const int64_t nt = g.ntm * g.ntn * p.nbatch;
  if (nt >= GRID_BLOCKS / 2) return hipErrorNotSupported;   // (its parts are fewer than as many again)
  const int64_t rest = nt % 256;
  g.S = tile_parts<T>(rest, BM, BN, p.T);
  g.part = nullptr;
  if (g.S > 1) {
    g.kc = ((p.T + g.S - 1) / g.S + TILE_K<T> - 1) / TILE_K<T> * TILE_K<T>;
    g.S = (int)((p.T + g.kc - 1) / g.kc);
    g.part = (T *)partials_alloc(sizeof(T) * (size_t)(rest * g.S * BM * BN));
    if (!g.part) g.S = 1;   // out of memory: whole tiles
  }
  g.nwhole = g.S > 1 ? nt - rest : nt;
  if (g.S == 1) g.kc = p.T;
  const bool ak = p.a_t == 1, bk = p.b_t == 1;
  const dim3 grid((unsigned)(g.nwhole + (nt - g.nwhole) * g.S));
  // (float) sums of 8 k rather than 32 where all of t is three stages or less;
  // up to half a stage, with the registers and LDS of that alone: eight blocks
  // per CU instead of four and half the matrix instructions (2000 products of
  // 100 x 8 x 100: 33 us against 50, 39 on the SIMT kernel, which also errs
  // 10% more; 20000 of 40 x 8 x 40: 64, 111 and 72; one of 15000 x 8 x 15000:
  // 232, 336 and 390)
  auto go = [&](auto how) {
    constexpr int F = decltype(how)::value;
    if (ak && bk) hipLaunchKernelGGL((tile_gemm<T, BM, BN, WR, WC, true, true, F>), grid, dim3(256), 0, s, a, b, c, g);
    else if (ak) hipLaunchKernelGGL((tile_gemm<T, BM, BN, WR, WC, true, false, F>), grid, dim3(256), 0, s, a, b, c, g);
    else if (bk) hipLaunchKernelGGL((tile_gemm<T, BM, BN, WR, WC, false, true, F>), grid, dim3(256), 0, s, a, b, c, g);
    else hipLaunchKernelGGL((tile_gemm<T, BM, BN, WR, WC, false, false, F>), grid, dim3(256), 0, s, a, b, c, g);
  };
  if constexpr (sizeof(T) == 4) {
    if (p.T <= TILE_K<T> / 2) go(std::integral_constant<int, HALF_STAGE>());
    else if (p.T <= 96) go(std::integral_constant<int, BY_EIGHT>());
    else go(std::integral_constant<int, BY_STAGE>());
  } else {
    go(std::integral_constant<int, BY_STAGE>());
  }
  if (g.part)
    hipLaunchKernelGGL((tile_join<T, BM, BN>), dim3((unsigned)((nt - g.nwhole) * (BM * BN / 256))), dim3(256), 0, s, c, g);
  const hipError_t e = hipGetLastError();
  if (g.part) partials_free(g.part);
  return e;
}

// 32 wide along a side where that saves a sixth of the padded width or more
static bool tile_narrow(int64_t n) { return 6 * ((n + 31) / 32 * 32) <= 5 * ((n + 63) / 64 * 64); }

template <class T> static hipError_t tile_T(const MmPlan &p, const T *a, const T *b, T *c, hipStream_t s) {
  // a side below 8 fills too little of a 16-wide instruction, fewer k too
  // little of a stage (double, 10 x 4 x 100, 3000 of them: 23.6 us, the SIMT
  // kernel 21.2)
  if (p.H < 8 || p.W < 8 || p.T < 8) return hipErrorNotSupported;
  if (tile_narrow(p.H)) {
    if (tile_narrow(p.W)) return tile_launch<T, 32, 32, 2, 2>(p, a, b, c, s);
    return tile_launch<T, 32, 64, 1, 4>(p, a, b, c, s);
  }
  if (tile_narrow(p.W) || p.variant == 32) return tile_launch<T, 64, 32, 4, 1>(p, a, b, c, s);
  return tile_launch<T, 64, 64, 2, 2>(p, a, b, c, s);
}

// Which engine runs a float product in the default mode: by its sizes alone, so
// that its bits depend neither on a timing nor on what ran before.  Batches
// have the kernel for 33..64 per side or the tiles; single products the tiles
// where the FP16 split's 128x128 blocks do not fit (a side below 64, or fewer
// than 32 k; 32 x 20000 x 20000 takes 395 us, on the SIMT kernel 4380), or
// where they are estimated to take no longer than the split, in us:
//   tiles  15 + operations / 92e6 + outputs / 2.2e6
//   split  50 + packed elements / 0.42e6 + outputs / 0.48e6 (stored, marked
//          and looked over), and 0.0175 per k for each 256 blocks of 128x128
// fitted to 140 products of 1.5e9 to 3e10 operations (standard deviations 10%
// and 8%; the choice is the faster engine's but for 2% to 9% on 8 of them).
// 1000^3: 31 and 69 us, 1587^3: 95 and 98, 2048^3: 170 and 115; 1000 x 6000 x
// 700: 105 and 165, 2500 x 1000 x 2500: 139 and 95.  Beyond 3e10 operations
// the split wins wherever it has blocks for the chip.
constexpr double SPLIT_FLOPS = 3e10;
bool tile_takes_f32(const MmPlan &p) {
  if (small_split16(p)) return false;
  const double h = (double)p.H, w = (double)p.W, k = (double)p.T, flops = 2.0 * h * w * k;
  if (!single_split16(p)) return true;
  if (flops > SPLIT_FLOPS) return false;
  const int64_t waves = ((p.H + 127) / 128 * ((p.W + 127) / 128) + 255) / 256;
  return 15 + flops / 92e6 + h * w / 2.2e6 <= 50 + (h + w) * k / 0.42e6 + h * w / 0.48e6 + 0.0175 * k * (double)waves;
}

// The widths of tile (MmPlan::variant) that the autotuner may choose from: 64
// and, where neither width is cut along t and so both sum every output alike,
// 64x32, which fills the chip better (600^3: 14 us against 21, 512^3: 12
// against 14) and reads more (3173 x 76 x 4691: 59 against 52).
std::vector<int> tile_widths_f32(const MmPlan &p) {
  const int64_t n32 = (p.H + 63) / 64 * ((p.W + 31) / 32), n64 = (p.H + 63) / 64 * ((p.W + 63) / 64);
  if (p.nbatch == 1 && !tile_narrow(p.H) && !tile_narrow(p.W) && tile_parts<float>(n64 % 256, 64, 64, p.T) == 1 &&
      tile_parts<float>(n32 % 256, 64, 32, p.T) == 1)
    return {64, 32};
  return {64};
}

hipError_t launch_tile_f64(const MmPlan &p, const double *a, const double *b, double *c, hipStream_t s) {
  return tile_T<double>(p, a, b, c, s);
}
hipError_t launch_tile_f32(const MmPlan &p, const float *a, const float *b, float *c, hipStream_t s) {
  return tile_T<float>(p, a, b, c, s);
}

}  // namespace pdlhip
