// Double matmult on v_mfma_f64_16x16x4_f64 in the default precision mode
// (lib/PDL/Primitive.pd:191-245: C[h][w] = sum_t A[h][t] B[t][w]).  FP64
// products and sums; lane l holds A[l%16][k] and B[k][l%16] for its k, and
// result register r of lane l is D[4r + l/16][l%16].
//
// Bound by the matrix cores (64 cycles per instruction), so the tiles are
// small: 64x64 of C per block of 4 waves keeps four blocks resident per CU,
// whose waves cover each other's loads and barriers, and cuts a product into
// enough blocks for 256 CUs.  4096^3: 2.09 ms, 65.8 TFLOP/s (128x128 blocks of
// the same kernel 2.33 ms, 128x64 2.28); 1500^3: 148 us (123 where the operands
// change from call to call; before, 144 blocks of 128x128: 280); 512^3: 18 us
// (the SIMT kernel: 85).  Operands go global -> registers -> LDS in stages of
// 16 k, two stages' loads in flight while the matrix cores work on a third
// (one: 59 instead of 54 us at 1024^3, where a CU has one block).  LDS holds
// rows of 16 k, padded to 18 doubles: a lane reads two neighbouring k of its
// row as 16 bytes (eight rows fall on distinct bank groups) and feeds them to
// two instructions; which k an instruction covers is free as long as A and B
// agree.
//
// Tiles that would fill only part of the chip in the last wave of blocks are
// cut along t into S parts, each summed into scratch, and joined by a second
// small kernel in a fixed order.
#include <hip/hip_runtime.h>

#include "device.hpp"
#include "launch.hpp"

namespace pdlhip {

void *scratch_alloc(size_t bytes);
void scratch_free(void *p);

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));
constexpr int DKB = 16, DKP = DKB + 2;

struct DgPlan {
  MmPlan p;
  int64_t ntm, ntn;    // tiles of one product
  int64_t nwhole;      // tiles summed over all of t; the others in S parts of kc
  int32_t S;
  int64_t kc;
  double *part;
};

// tile t of all products -> product, tile row, tile column: groups of 8 tile
// rows column by column, for the L2's sake
__device__ inline void dg_tile(const DgPlan &g, int64_t t, int64_t *o, int64_t &tm, int64_t &tn) {
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

// One operand's share of a stage: N rows x 16 k as N * 8 pairs of k over 256
// threads.  KFAST (unit stride along t): neighbouring threads take
// neighbouring pairs, a pair per load (16 bytes, which the hardware takes at
// any 8-byte address); else neighbouring threads take neighbouring rows.  The
// first stage takes the k that do not fill a stage (or 16), so that the loop's
// loads are whole, sit behind no branch, and their waits are counted.
template <int N, bool KFAST> struct DgLoad {
  static constexpr int P = N * 8 / 256;
  typedef d2 __attribute__((aligned(8))) d2u;
  gptr<const double> ptr[P];   // (stated global: a generic pointer would load through the flat path)
  d2 v[2][P];                  // two stages on their way
  __device__ static int row(int s) { const int e = threadIdx.x + 256 * s; return KFAST ? e / 8 : e % N; }
  __device__ static int pair(int s) { const int e = threadIdx.x + 256 * s; return KFAST ? e % 8 : e / N; }
  // the first stage's `some` k, zeros after them, into l; rows past the
  // operand's last repeat it: they reach only outputs that are not stored
  __device__ void first(const double *base, int64_t r0, int64_t R, int64_t inc_r, int64_t k0, int64_t inc_k, int some,
                        double (*l)[DKP]) {
#pragma unroll
    for (int s = 0; s < P; s++) {
      const int64_t r = r0 + row(s) < R ? r0 + row(s) : R - 1;
      const int k = 2 * pair(s);
      ptr[s] = as_global(base + r * inc_r + (k0 + k) * inc_k);
      v[0][s] = d2{k < some ? ptr[s][0] : 0.0, k + 1 < some ? ptr[s][inc_k] : 0.0};
    }
    stage(0, l);
#pragma unroll
    for (int s = 0; s < P; s++) ptr[s] += some * inc_k;
  }
  // the stage at ptr, which moves on if another follows
  __device__ void load(int set, int64_t inc_k, bool more) {
#pragma unroll
    for (int s = 0; s < P; s++) {
      if (KFAST) v[set][s] = *(gptr<const d2u>)ptr[s];
      else v[set][s] = d2{ptr[s][0], ptr[s][inc_k]};
    }
    const int64_t step = more ? DKB * inc_k : 0;
#pragma unroll
    for (int s = 0; s < P; s++) ptr[s] += step;
  }
  __device__ void stage(int set, double (*l)[DKP]) {
#pragma unroll
    for (int s = 0; s < P; s++) *reinterpret_cast<d2 *>(&l[row(s)][2 * pair(s)]) = v[set][s];
  }
};

template <int BM, int BN, int WR, int WC, bool AK, bool BK>
__global__ __launch_bounds__(256, 4) void dgemm(const double *__restrict__ a, const double *__restrict__ b,
                                             double *__restrict__ c, DgPlan g) {
  constexpr int TI = BM / WR / 16, TJ = BN / WC / 16;
  static_assert(WR * WC == 4, "four waves");
  __shared__ __align__(16) double sA[2][BM][DKP];
  __shared__ __align__(16) double sB[2][BN][DKP];
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
  dg_tile(g, t, o, tm, tn);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wr = w / WC, wc = w % WC, fr = lane & 15, fk = lane >> 4;
  const int64_t m0 = tm * BM, n0 = tn * BN;
  DgLoad<BM, AK> la;
  DgLoad<BN, BK> lb;
  const int some = (int)((ke - kb - 1) % DKB) + 1;
  const int64_t n = (ke - kb - some) / DKB + 1;   // stages
  la.first(a + o[0], m0, p.H, p.a_h, kb, p.a_t, some, sA[0]);
  lb.first(b + o[1], n0, p.W, p.b_w, kb, p.b_t, some, sB[0]);
  d4 acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; i++)
#pragma unroll
    for (int j = 0; j < TJ; j++) acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};
  // A step multiplies the two halves of its 16 k.  The barrier stands between
  // them: before it the next stage goes to the other buffer (whose last
  // reads came before the barrier of the step before) and the second half's
  // fragments are read, after it the next step's first half, so that every
  // LDS read has a half's matrix instructions to arrive in.
  auto fetch = [&](int set, int64_t q) {   // stage q (past the last one, that again, unused)
    la.load(set, p.a_t, q + 1 < n);
    lb.load(set, p.b_t, q + 1 < n);
  };
  d2 af[2][TI], bf[2][TJ];
  auto frags = [&](int half, int buf) {
#pragma unroll
    for (int i = 0; i < TI; i++)
      af[half][i] = *reinterpret_cast<const d2 *>(&sA[buf][(wr * TI + i) * 16 + fr][half * 8 + 2 * fk]);
#pragma unroll
    for (int j = 0; j < TJ; j++)
      bf[half][j] = *reinterpret_cast<const d2 *>(&sB[buf][(wc * TJ + j) * 16 + fr][half * 8 + 2 * fk]);
  };
  auto multiply = [&](int half) {
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[half][i][u], bf[half][j][u], acc[i][j], 0, 0, 0);
  };
  auto step = [&](int cur, int64_t q) {   // multiplies stage q, in buffer cur; set cur ^ 1 holds the next one
    la.stage(cur ^ 1, sA[cur ^ 1]);
    lb.stage(cur ^ 1, sB[cur ^ 1]);
    fetch(cur ^ 1, q + 3);
    frags(1, cur);
    __builtin_amdgcn_sched_barrier(0);   // the compiler sinks the reads to their uses otherwise
    multiply(0);
    __syncthreads();
    frags(0, cur ^ 1);
    __builtin_amdgcn_sched_barrier(0);
    multiply(1);
  };
  auto last_step = [&](int cur) {
    frags(1, cur);
    multiply(0);
    multiply(1);
  };
  if (n > 1) {
    fetch(1, 1);
    fetch(0, 2);
  }
  __syncthreads();
  frags(0, 0);
  int64_t q = 0;
  for (; q + 2 < n; q += 2) {
    step(0, q);
    step(1, q + 1);
  }
  if (q + 1 < n) {
    step(0, q);
    last_step(1);
  } else {
    last_step(0);
  }
#pragma unroll
  for (int i = 0; i < TI; i++)
#pragma unroll
    for (int j = 0; j < TJ; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int h = (wr * TI + i) * 16 + 4 * r + fk, wv = (wc * TJ + j) * 16 + fr;
        if (part >= 0)
          g.part[(((t - g.nwhole) * g.S + part) * BM + h) * BN + wv] = acc[i][j][r];
        else if (m0 + h < p.H && n0 + wv < p.W)
          c[o[2] + (n0 + wv) * p.c_w + (m0 + h) * p.c_h] = acc[i][j][r];
      }
}

// the parts of each cut tile, added in ascending t
template <int BM, int BN>
__global__ __launch_bounds__(256) void dgemm_join(double *__restrict__ c, DgPlan g) {
  constexpr int PER = BM * BN / 256;
  const int64_t q = blockIdx.x / PER;
  const int e = (int)(blockIdx.x % PER) * 256 + threadIdx.x, h = e / BN, wv = e % BN;
  const double *src = g.part + q * g.S * (BM * BN) + e;
  double s = src[0];
  for (int k = 1; k < g.S; k++) s += src[(int64_t)k * (BM * BN)];
  int64_t o[3], tm, tn;
  dg_tile(g, g.nwhole + q, o, tm, tn);
  if (tm * BM + h < g.p.H && tn * BN + wv < g.p.W)
    c[o[2] + (tn * BN + wv) * g.p.c_w + (tm * BM + h) * g.p.c_h] = s;
}

template <int BM, int BN, int WR, int WC>
static hipError_t dgemm_launch(const MmPlan &p, const double *a, const double *b, double *c, hipStream_t s) {
  DgPlan g;
  g.p = p;
  g.ntm = (p.H + BM - 1) / BM;
  g.ntn = (p.W + BN - 1) / BN;
  const int64_t nt = g.ntm * g.ntn * p.nbatch;
  if (nt >= ((int64_t)1 << 30)) return hipErrorNotSupported;
  // Tiles past the last multiple of 256 (a tile per CU) leave CUs idle for a
  // whole tile's time.  Cutting each into S parts makes that ceil(rest * S /
  // 256) / S of it, for a second launch and the parts' traffic (about 4 us);
  // a part keeps at least 64 k.
  constexpr double CU_FLOPS = 0.24e6;   // per us and CU, as measured
  const int64_t rest = nt % 256;
  const double tile_us = 2.0 * BM * BN * (double)p.T / CU_FLOPS;
  g.S = 1;
  double best = rest ? tile_us : 0.0;
  for (int S = 2; S <= 16 && rest && p.T / S >= 64; S++) {
    const double us = tile_us * (double)((rest * S + 255) / 256) / S + 4.0 + (double)(rest * S * BM * BN * 16) / 3e6;
    if (us < best) { best = us; g.S = S; }
  }
  g.part = nullptr;
  if (g.S > 1) {
    g.kc = ((p.T + g.S - 1) / g.S + DKB - 1) / DKB * DKB;
    g.S = (int)((p.T + g.kc - 1) / g.kc);
    g.part = (double *)scratch_alloc(sizeof(double) * (size_t)(rest * g.S * BM * BN));
    if (!g.part) g.S = 1;   // none cached during a capture: whole tiles
  }
  g.nwhole = g.S > 1 ? nt - rest : nt;
  if (g.S == 1) g.kc = p.T;
  const bool ak = p.a_t == 1, bk = p.b_t == 1;
  const dim3 grid((unsigned)(g.nwhole + (nt - g.nwhole) * g.S));
  if (ak && bk) hipLaunchKernelGGL((dgemm<BM, BN, WR, WC, true, true>), grid, dim3(256), 0, s, a, b, c, g);
  else if (ak) hipLaunchKernelGGL((dgemm<BM, BN, WR, WC, true, false>), grid, dim3(256), 0, s, a, b, c, g);
  else if (bk) hipLaunchKernelGGL((dgemm<BM, BN, WR, WC, false, true>), grid, dim3(256), 0, s, a, b, c, g);
  else hipLaunchKernelGGL((dgemm<BM, BN, WR, WC, false, false>), grid, dim3(256), 0, s, a, b, c, g);
  if (g.part)
    hipLaunchKernelGGL((dgemm_join<BM, BN>), dim3((unsigned)((nt - g.nwhole) * (BM * BN / 256))), dim3(256), 0, s, c, g);
  const hipError_t e = hipGetLastError();
  if (g.part) scratch_free(g.part);
  return e;
}

hipError_t launch_mfma_f64(const MmPlan &p, const double *a, const double *b, double *c, hipStream_t s) {
  // a side below 8 fills too little of a 16-wide instruction, fewer k too
  // little of a stage (10 x 4 x 100, 3000 of them: 23.6 us, the SIMT kernel 21.2)
  if (p.H < 8 || p.W < 8 || p.T < 8) return hipErrorNotSupported;
  // 32 wide along a side where that saves a sixth of the padded width or more
  auto narrow = [](int64_t n) { return 6 * ((n + 31) / 32 * 32) <= 5 * ((n + 63) / 64 * 64); };
  if (narrow(p.H)) {
    if (narrow(p.W)) return dgemm_launch<32, 32, 2, 2>(p, a, b, c, s);
    return dgemm_launch<32, 64, 1, 4>(p, a, b, c, s);
  }
  if (narrow(p.W)) return dgemm_launch<64, 32, 4, 1>(p, a, b, c, s);
  return dgemm_launch<64, 64, 2, 2>(p, a, b, c, s);
}

}  // namespace pdlhip
