// The matrix-core product of the split-FP16 mode (k_mfma.hip packs the
// operands and recomputes what the split cannot hold): per 16-deep k slice
// and pair of 32x32 tiles three v_mfma_f32_32x32x16_f16, lo*hi + hi*lo +
// hi*hi, accumulated in FP32.
#include <hip/hip_runtime.h>

#include "launch.hpp"
#include "mfma_common.hpp"

namespace pdlhip {

// BM x BN of C per block of WR x WC waves, TI x TJ tiles of 32x32 per wave.
// k slices of 16 stream through a ring of HG_SLOTS slots in LDS.  At slice i
// a wave waits for its own loads of slice i + 1, meets the others at the
// barrier (which also says that slot i - 1 has been read by all), refills
// that slot, reads slice i + 1's fragments into the register set that slice
// i - 1 used, and multiplies slice i.  So loads have three slices' time to
// arrive and LDS reads one, and each slice costs one barrier.
//
// Bound by the matrix cores and, with random data, by the power they draw:
// 8192^3 takes 2.6 ms (1276 TFLOP/s of FP16; a library FP16 product of the
// size 1150 to 1460 by layout), zeros 1.9.  With two stages of 32 k, a full
// wait for the loads at each barrier and LDS reads after it: 3.1 to 3.2 ms.
// Matrix instructions first and memory accesses between them gained the most;
// 128x128 blocks take 3.3 ms there and win below about 1024 a side.
constexpr int HG_SLOTS = 5;

template <int BM, int BN, int WR, int WC>
__global__ __launch_bounds__(WR * WC * 64, 2) void split16_gemm(const half_t *__restrict__ A,
                                                                const half_t *__restrict__ B,
                                                                const float *__restrict__ sA,
                                                                const float *__restrict__ sB,
                                                                const float *__restrict__ dA,
                                                                const float *__restrict__ dB, int *rowflag,
                                                                float *__restrict__ c, MmPlan p, int nk, int64_t ntm,
                                                                int64_t ntn) {
  constexpr int NW = WR * WC, TI = BM / WR / 32, TJ = BN / WC / 32;
  constexpr int GA = BM / 32, GB = BN / 32, NP = 2 * (GA + GB);   // row groups, pieces of a slice
  constexpr int ND = NP / NW;                                       // pieces each wave brings in
  static_assert(NP % NW == 0 && ND == 4, "the waits below count four loads per slice");
  __shared__ __align__(16) half_t lds[HG_SLOTS][NP][PIECE];
  int64_t tm, tn;
  tile_of(blockIdx.x, ntm, ntn, tm, tn);
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = w / WC, wc = w % WC;
  const half_t *src[ND];
#pragma unroll
  for (int d = 0; d < ND; d++) {
    const int q = w * ND + d, g = q >> 1;   // piece: A's row groups, then B's, hi and lo of each
    const half_t *base = g < GA ? A + (tm * GA + g) * (int64_t)nk * (2 * PIECE) : B + (tn * GB + g - GA) * (int64_t)nk * (2 * PIECE);
    src[d] = base + (q & 1) * PIECE + lane * 8;
  }
  auto bring = [&](int d, int slot, int ks) {   // (past the last slice, that one again, unused)
    const int64_t k = ks < nk ? ks : nk - 1;
    dma16(src[d] + k * (2 * PIECE), &lds[slot][w * ND + d][0]);
  };
  // 32x32x16 operand layout: lane l holds row (l % 32), k (l / 32) * 8 .. +7
  const int lr = lane & 31, at = lr * 16 + (((lane >> 5) ^ (lr >> 2 & 1)) * 8);
  constexpr int NF = 2 * (TI + TJ);   // fragments of a slice: B's column tiles hi and lo, then A's rows
  half8 f[2][NF];
  auto frag = [&](int set, int n, int slot) {
    const int q = n < 2 * TJ ? 2 * (GA + wc * TJ) + n : 2 * (wr * TI) + n - 2 * TJ;
    f[set][n] = *reinterpret_cast<const half8 *>(&lds[slot][q][at]);
  };
  f32x16 acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; i++)
#pragma unroll
    for (int j = 0; j < TJ; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
  // matrix instruction m of a slice: per row tile the products lo*hi, hi*lo
  // and hi*hi, each over the row's TJ accumulators
  constexpr int NM = 3 * TI * TJ;
  auto mfma = [&](int set, int m) {
    const int i = m / (3 * TJ), x = m / TJ % 3, j = m % TJ;
    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[set][2 * TJ + 2 * i + (x == 0)], f[set][2 * j + (x == 1)],
                                                        acc[i][j], 0, 0, 0);
  };
  auto meet = [&] {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
#pragma unroll
  for (int k = 0; k < HG_SLOTS - 1; k++)
#pragma unroll
    for (int d = 0; d < ND; d++) bring(d, k, k);
  __builtin_amdgcn_s_waitcnt(0x0f7c);   // vmcnt(12): slice 0 of this wave's four
  meet();
#pragma unroll
  for (int n = 0; n < NF; n++) frag(0, n, 0);
  int slot = 0;   // of slice i
  // one memory access after each of the first matrix instructions, which
  // execute meanwhile; left to itself the compiler puts all of them first
  static_assert(NM >= ND + NF, "a matrix instruction per access");
  auto step = [&](int set, int i) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0078);   // vmcnt(8) lgkmcnt(0): slices i + 2 and i + 3 may still be on their way
    meet();
    const int old = slot == 0 ? HG_SLOTS - 1 : slot - 1;
    slot = slot == HG_SLOTS - 1 ? 0 : slot + 1;
#pragma unroll
    for (int m = 0; m < NM; m++) {
      mfma(set, m);
      if (m < ND) bring(m, old, i + HG_SLOTS - 1);
      else if (m < ND + NF) frag(set ^ 1, m - ND, slot);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  int i = 0;
  for (; i + 1 < nk; i += 2) {
    step(0, i);
    step(1, i + 1);
  }
  if (i < nk) {
#pragma unroll
    for (int m = 0; m < NM; m++) mfma(0, m);
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): no load to LDS outlives the block
  // D layout of a 32x32 tile: lane l, reg r -> row 8*(r/4) + 4*(l/32) + r%4, col l%32
#pragma unroll
  for (int ti = 0; ti < TI; ti++)
#pragma unroll
    for (int tj = 0; tj < TJ; tj++)
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const int64_t h = tm * BM + (wr * TI + ti) * 32 + 8 * (r / 4) + 4 * (lane >> 5) + (r & 3);
        const int64_t wcol = tn * BN + (wc * TJ + tj) * 32 + (lane & 31);
        if (h < p.H && wcol < p.W)
          c[p.off[2] + wcol * p.c_w + h * p.c_h] = mm_finish(acc[ti][tj][r], dA[h], dB[wcol], sA[h], sB[wcol], rowflag, h);
      }
}

hipError_t launch_split16(bool big, const half_t *A, const half_t *B, const float *sA, const float *sB, const float *dA,
                          const float *dB, int *rowflag, float *c, const MmPlan &p, int64_t Kp, int64_t ntm, int64_t ntn,
                          hipStream_t s) {
  const dim3 grid((unsigned)(ntm * ntn));
  if (big)
    hipLaunchKernelGGL((split16_gemm<256, 256, 4, 2>), grid, dim3(512), 0, s, A, B, sA, sB, dA, dB, rowflag, c, p,
                       (int)(Kp / 16), ntm, ntn);
  else
    hipLaunchKernelGGL((split16_gemm<128, 128, 2, 2>), grid, dim3(256), 0, s, A, B, sA, sB, dA, dB, rowflag, c, p,
                       (int)(Kp / 16), ntm, ntn);
  return hipGetLastError();
}

}  // namespace pdlhip
