// Lists of uneven matmults in one launch (the reference runs such a list as a
// Perl loop of matmult calls, lib/PDL/Primitive.pd:197-209 per item).  The
// host builds one work item per (product, C tile), ordered by decreasing
// inner dimension (longest-processing-time first).  Float and double lists in
// the default modes run on the matrix cores (list_tiles).  PDL order and the integer types run the SIMT tile of
// k_matmult.hip (accumulation order per output: ascending t, so the PDL-order
// variant stays bit-identical to PDL's loop) in persistent blocks, which take
// items from a device counter until the queue is drained, so every block
// reaches the exit condition; so does the BF16 split.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device.hpp"
#include "launch.hpp"
#include "mm_tile.hpp"

namespace pdlhip {

template <class T, bool FUSED, int TS>
__device__ inline void list_tile(const MmItem &it, int64_t tm, int64_t tn, T (*As)[TS + 1], T (*Bs)[TS + 1]) {
  constexpr int KS = 16;
  constexpr int PT = TS / 16;          // outputs per thread per dim (16x16 threads)
  const T *a = (const T *)it.a, *b = (const T *)it.b;
  T *c = (T *)it.c;
  const int tid = threadIdx.x, tx = tid % 16, ty = tid / 16;
  const int64_t h0 = tm * TS, w0 = tn * TS;
  T acc[PT][PT];
#pragma unroll
  for (int i = 0; i < PT; i++)
#pragma unroll
    for (int j = 0; j < PT; j++) acc[i][j] = T(0);
  constexpr int NE = TS * KS / 256;   // staged elements per thread per operand
  for (int64_t k0 = 0; k0 < it.T; k0 += KS) {
    // every load of the chunk is issued before the first LDS write; indices
    // are clamped into the operand and the element zeroed afterwards, so no
    // load sits behind a branch
    T ra[NE], rb[NE];
#pragma unroll
    for (int q = 0; q < NE; q++) {
      const int e = tid + 256 * q;
      const int kk = e % KS, mm = e / KS, nn = e % TS, kb = e / TS;
      const int64_t gh = h0 + mm, gt = k0 + kk, gw = w0 + nn, gt2 = k0 + kb;
      const int64_t ch = gh < it.H ? gh : it.H - 1, ct = gt < it.T ? gt : it.T - 1;
      const int64_t cw = gw < it.W ? gw : it.W - 1, ct2 = gt2 < it.T ? gt2 : it.T - 1;
      ra[q] = a[it.oa + ct * it.a_t + ch * it.a_h];
      rb[q] = b[it.ob + cw * it.b_w + ct2 * it.b_t];
    }
#pragma unroll
    for (int q = 0; q < NE; q++) {
      const int e = tid + 256 * q;
      const int kk = e % KS, mm = e / KS, nn = e % TS, kb = e / TS;
      As[kk][mm] = (h0 + mm < it.H && k0 + kk < it.T) ? ra[q] : T(0);
      Bs[kb][nn] = (w0 + nn < it.W && k0 + kb < it.T) ? rb[q] : T(0);
    }
    __syncthreads();
    const int kmax = (it.T - k0 < KS) ? (int)(it.T - k0) : KS;
    for (int kk = 0; kk < kmax; kk++) {
      T av[PT], bv[PT];
#pragma unroll
      for (int i = 0; i < PT; i++) av[i] = As[kk][ty + 16 * i];
#pragma unroll
      for (int j = 0; j < PT; j++) bv[j] = Bs[kk][tx + 16 * j];
#pragma unroll
      for (int i = 0; i < PT; i++)
#pragma unroll
        for (int j = 0; j < PT; j++) {
          if constexpr (FUSED && IsFloat<T>::v) acc[i][j] = fma(av[i], bv[j], acc[i][j]);
          else acc[i][j] = wadd(acc[i][j], wmul(av[i], bv[j]));
        }
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < PT; i++) {
    int64_t gh = h0 + ty + 16 * i;
    if (gh >= it.H) continue;
#pragma unroll
    for (int j = 0; j < PT; j++) {
      int64_t gw = w0 + tx + 16 * j;
      if (gw < it.W) c[it.oc + gw * it.c_w + gh * it.c_h] = acc[i][j];
    }
  }
}

// The work list holds LIST_BINS bins back to back, bin x = work[bounds[x]
// .. bounds[x + 1]), one per XCD: the host spreads the products over the
// bins by their work (largest first, each to the lightest bin), so all the
// tiles of a product sit in one bin, in order.  Workgroups go to the 8 XCDs
// round-robin, so block b starts on bin b % 8 and the tiles of a product,
// taken by neighbouring blocks of one XCD at about the same time, re-read
// its A and B panels from that XCD's L2 rather than from HBM; a block whose
// bin is empty goes on to the next bins.  counter[x * LIST_CSTRIDE] is bin
// x's counter, each in a 128-byte line of its own (reset by a kernel before
// each launch); the bounds follow the counters.
constexpr int LIST_BINS = 8, LIST_CSTRIDE = 32, LIST_BOUNDS = LIST_BINS * LIST_CSTRIDE;

__global__ void list_reset(unsigned int *counter) {
  if (threadIdx.x < LIST_BINS && blockIdx.x == 0) counter[threadIdx.x * LIST_CSTRIDE] = 0u;
}

// the block's next work item (false: every bin is empty); thread 0 takes it
// and hands it on through LDS
__device__ __forceinline__ bool list_next(unsigned int *counter, const unsigned int *__restrict__ bounds,
                                          const int3 *__restrict__ work, int &bin, unsigned &done, unsigned *sh,
                                          int3 &job) {
  if (threadIdx.x == 0) {
    unsigned w = ~0u;
    while (done != (1u << LIST_BINS) - 1u) {
      const unsigned i = atomicAdd(counter + bin * LIST_CSTRIDE, 1u);
      if (bounds[bin] + i < bounds[bin + 1]) {
        w = bounds[bin] + i;
        break;
      }
      done |= 1u << bin;
      bin = (bin + 1) % LIST_BINS;
    }
    *sh = w;
  }
  __syncthreads();
  const unsigned w = *sh;
  __syncthreads();
  if (w == ~0u) return false;
  job = work[w];
  return true;
}

// persistent: take work items until every bin is empty
template <class T, bool FUSED, int TS>
__global__ __launch_bounds__(256) void list_queue(const MmItem *__restrict__ items, const int3 *__restrict__ work,
                                                  const unsigned int *__restrict__ bounds, unsigned int *counter) {
  constexpr int KS = 16;
  __shared__ T As[KS][TS + 1];
  __shared__ T Bs[KS][TS + 1];
  __shared__ unsigned int next;
  int bin = blockIdx.x % LIST_BINS;
  unsigned done = 0;
  int3 job;
  while (list_next(counter, bounds, work, bin, done, &next, job))
    list_tile<T, FUSED, TS>(items[job.x], job.y, job.z, As, Bs);
}

// one launch per item (the comparison the list path is measured against)
template <class T, bool FUSED, int TS>
__global__ __launch_bounds__(256) void list_one(const MmItem *__restrict__ items, int idx, int64_t ntn) {
  constexpr int KS = 16;
  __shared__ T As[KS][TS + 1];
  __shared__ T Bs[KS][TS + 1];
  list_tile<T, FUSED, TS>(items[idx], blockIdx.x / ntn, blockIdx.x % ntn, As, Bs);
}

// ---------------------------------------------------------------- matrix cores
// Float and double lists in the default modes run on the matrix cores with
// FP32 / FP64 products and sums: the instructions, stages and LDS rows of
// mm_tile.hpp (float: partial sums of 32 k), TS x TS of C per work item.
//
// A tile lasts only a few stages, so a tile by itself is bound by the chain
// it waits for: its work item, its operands' addresses, its first stages, one
// memory latency each.  So a block runs through its work items as one
// sequence of stages: two stages' loads are in flight while a third is
// multiplied, also across the end of a tile.  Every fetch issues the same
// loads whatever the tile's sizes (past the last stage, that stage again), so
// that their waits stay counted: rows past an operand's last repeat it, and a
// first stage of fewer k loads a whole one, or from the last k where that fits,
// and is zeroed on its way to LDS.  A wave's 16x16 tiles lie 32 apart, so that where
// no more than 32 rows or columns are inside the product each of the four
// skips half of its instructions.
//
// Block b runs on XCD b % 8 and takes one item of each round of grid / 8 items
// of bin b % 8, largest inner dimension first, so that the blocks' shares
// differ little: the b / 8th of the first round and one five places on in each
// next, lest a block meet the edge tiles of one product after the other.
//
// 4096 float products of 8..256 per side: 547 us (a tile at a time, taken from
// a counter: 621; a workgroup per tile: 662), 63 TFLOP/s of the products' own
// operations, 75 with the padding; double 937 (978).  300 of 8..64: 7.2 us
// (14.5), 64 of 8..256: 14.9 (28.8), where the counter's latency was most of
// it.  Four blocks per CU (without the partial sums) take as long as three,
// and products of 256 alone reach 82 TFLOP/s: what is left is the LDS and
// vector work between matrix instructions, about as long as those.
typedef float lf32x16 __attribute__((ext_vector_type(16)));

template <int TS> constexpr int LIST_PER_CU = TS == 32 ? 6 : 3;

// one operand's loads: thread t takes group % 8 of row / 8 (KFAST) or row t %
// TS, as TileLoad does
template <class T, int TS, bool KFAST> struct ListLoad {
  static constexpr int P = TS * 8 / 256, V = TILE_V<T>, KB = TILE_K<T>;
  typedef typename TileType<T>::vec_t vec;
  typedef vec __attribute__((aligned(sizeof(T)))) vecu;
  gptr<const T> at[P];   // the thread's k of the stage
  int64_t inc_k;
  vec v[2][P];
  __device__ static int row(int s) { const int e = threadIdx.x + 256 * s; return KFAST ? e / 8 : e % TS; }
  __device__ static int group(int s) { const int e = threadIdx.x + 256 * s; return KFAST ? e % 8 : e / TS; }
  // `top`: the last k at which V of them can be loaded (KB: anywhere in a stage)
  __device__ __forceinline__ void open(const T *base, int r0, int R, int64_t inc_r, int64_t ik, int top) {
#pragma unroll
    for (int s = 0; s < P; s++) {
      const int r = r0 + row(s) < R ? r0 + row(s) : R - 1;
      const int k = V * group(s);
      at[s] = as_global(base + r * inc_r + (k < top ? k : top) * ik);
    }
    inc_k = ik;
  }
  // a stage's loads; `most`: the last of the V that there is (strided only)
  __device__ __forceinline__ void load(int set, int most) {
#pragma unroll
    for (int s = 0; s < P; s++) {
      if (KFAST) v[set][s] = *(gptr<const vecu>)at[s];
      else
#pragma unroll
        for (int i = 0; i < V; i++) v[set][s][i] = at[s][(i < most ? i : most) * inc_k];
    }
  }
  __device__ __forceinline__ void advance(int k) {
#pragma unroll
    for (int s = 0; s < P; s++) at[s] += k * inc_k;
  }
  // zero from `some` k on; what was loaded from `top` instead of the group's
  // own k goes back to its place
  __device__ __forceinline__ void stage(int set, int some, int top, T (*l)[TILE_P<T>]) {
    if (some < KB) {
#pragma unroll
      for (int s = 0; s < P; s++) {
        const int k = V * group(s), d = k < top ? 0 : k - top;
        vec x;
#pragma unroll
        for (int i = 0; i < V; i++) {
          x[i] = T(0);
#pragma unroll
          for (int j = i; j < V; j++) x[i] = d == j - i ? v[set][s][j] : x[i];
          x[i] = i < some - k ? x[i] : T(0);
        }
        v[set][s] = x;
      }
    }
#pragma unroll
    for (int s = 0; s < P; s++) *reinterpret_cast<vec *>(&l[row(s)][V * group(s)]) = v[set][s];
  }
};

// `work` null: the tiles of product `only`, ntn of them a row, one a block
template <class T, int TS, bool AK, bool BK>
__global__ __launch_bounds__(256, LIST_PER_CU<TS>) void list_tiles(const MmItem *__restrict__ items,
                                                                    const int3 *__restrict__ work,
                                                                    const unsigned int *__restrict__ bounds, int only,
                                                                    unsigned ntn) {
  constexpr int KB = TILE_K<T>, V = TILE_V<T>, TI = TS / 32;
  // of a stage: ends its tile; more than 32 rows, columns of it inside the
  // product; more than half of its k
  constexpr unsigned LAST = 1, HIGH = 2, WIDE = 4, DEEP = 8, KIND = 4;
  typedef TileType<T> TT;
  __shared__ __align__(16) T sA[2][TS][TILE_P<T>];
  __shared__ __align__(16) T sB[2][TS][TILE_P<T>];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wr = w >> 1, wc = w & 1, fr = lane & 15, fk = lane >> 4;
  const unsigned bin = blockIdx.x % LIST_BINS, step = work ? gridDim.x / LIST_BINS : gridDim.x;
  const unsigned end = work ? bounds[bin + 1] : gridDim.x, turn = 5 % step;
  struct Place {
    unsigned round, slot;
    __device__ unsigned at() const { return round + slot; }
  };
  auto after = [&](Place p) {
    const unsigned slot = p.slot + turn;
    return Place{p.round + step, slot < step ? slot : slot - step};
  };
  Place lw = {work ? bounds[bin] : 0, work ? blockIdx.x / LIST_BINS : blockIdx.x}, cw = lw;   // loaded, multiplied item
  if (lw.at() >= end) return;
  auto job_at = [&](unsigned i) { return work ? work[i] : make_int3(only, (int)(i / ntn), (int)(i % ntn)); };
  ListLoad<T, TS, AK> la;
  ListLoad<T, TS, BK> lb;
  // the loaded item: stages left, the first one's k, HIGH and WIDE, and for
  // its loads: the last k for a whole group, the last of a group's k
  int left = 0, first = 0, top = 0, most = 0;
  unsigned sides = 0;
  auto open = [&]() {
    const int3 job = job_at(lw.at());
    const MmItem &it = items[job.x];
    const int K = (int)it.T;
    const bool any = K > 0;   // an empty inner dimension: one stage of zeros, its loads from the item table
    left = any ? (K - 1) / KB + 1 : 1;
    first = any ? (K - 1) % KB + 1 : 0;
    top = K >= KB ? KB : K > V ? K - V : 0;
    most = K >= V ? V - 1 : any ? K - 1 : 0;
    la.open(any ? (const T *)it.a + it.oa : (const T *)items, any ? job.y * TS : 0, any ? (int)it.H : 1,
            it.a_h, any ? it.a_t : 0, top);
    lb.open(any ? (const T *)it.b + it.ob : (const T *)items, any ? job.z * TS : 0, any ? (int)it.W : 1,
            it.b_w, any ? it.b_t : 0, top);
    sides = ((int)it.H - job.y * TS > 32 ? HIGH : 0) | ((int)it.W - job.z * TS > 32 ? WIDE : 0);
  };
  int some[2], tops[2];   // of the stages in the two register sets
  unsigned kinds = 0;     // of the stages ahead, KIND bits each
  int ahead = 0;
  bool fresh = true;
  auto fetch = [&](int set) {
    if (left == 0 && after(lw).at() < end) {
      lw = after(lw);
      open();
      fresh = true;
    }
    la.load(set, most);
    lb.load(set, most);
    some[set] = fresh ? first : KB;
    tops[set] = top;
    kinds |= (sides | (left == 1 ? LAST : 0) | (some[set] > KB / 2 ? DEEP : 0)) << (KIND * ahead);
    const int go = left > 1 ? some[set] : 0;
    la.advance(go);
    lb.advance(go);
    fresh = false;
    if (left > 0) left--;
  };
  typename TT::acc_t acc[TI][TI], part[TI][TI];
  typename TT::vec_t af[2][TI], bf[2][TI];
  auto clear = [&]() {
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
      for (int j = 0; j < TI; j++) acc[i][j] = part[i][j] = typename TT::acc_t{T(0), T(0), T(0), T(0)};
  };
  auto frags = [&](int half, int buf) {
#pragma unroll
    for (int i = 0; i < TI; i++)
      af[half][i] = *reinterpret_cast<const typename TT::vec_t *>(&sA[buf][(2 * i + wr) * 16 + fr][half * KB / 2 + V * fk]);
#pragma unroll
    for (int j = 0; j < TI; j++)
      bf[half][j] = *reinterpret_cast<const typename TT::vec_t *>(&sB[buf][(2 * j + wc) * 16 + fr][half * KB / 2 + V * fk]);
  };
  auto mult = [&](int half, int ni, int nj) {
#pragma unroll
    for (int u = 0; u < V; u++)
#pragma unroll
      for (int i = 0; i < ni; i++)
#pragma unroll
        for (int j = 0; j < nj; j++) {
          if constexpr (sizeof(T) == 8) {
            acc[i][j] = TT::mfma(af[half][i][u], bf[half][j][u], acc[i][j]);
          } else {
            if (half == 0 && u == 0) acc[i][j] += part[i][j];
            part[i][j] = TT::mfma(af[half][i][u], bf[half][j][u], half == 0 && u == 0 ? typename TT::acc_t{} : part[i][j]);
          }
        }
  };
  auto multiply = [&](int half) {
    if (half == 1 && !(kinds & DEEP)) return;
    if constexpr (TI == 1) {
      mult(half, 1, 1);
    } else if (kinds & HIGH) {
      if (kinds & WIDE) mult(half, 2, 2);
      else mult(half, 2, 1);
    } else {
      if (kinds & WIDE) mult(half, 1, 2);
      else mult(half, 1, 1);
    }
  };
  auto store = [&]() {
    const int3 job = job_at(cw.at());
    const MmItem &it = items[job.x];
    const int64_t m0 = (int64_t)job.y * TS, n0 = (int64_t)job.z * TS, c_h = it.c_h, c_w = it.c_w;
    const int rows = (int)(it.H - m0 < TS ? it.H - m0 : TS), cols = (int)(it.W - n0 < TS ? it.W - n0 : TS);
    const auto c = as_global((T *)it.c + it.oc + m0 * c_h + n0 * c_w);
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
      for (int j = 0; j < TI; j++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int h = (2 * i + wr) * 16 + TT::row(r, fk), n = (2 * j + wc) * 16 + fr;
          T v = acc[i][j][r];
          if constexpr (sizeof(T) == 4) v += part[i][j][r];
          if (h < rows && n < cols) c[h * c_h + n * c_w] = v;
        }
  };
  // multiplies the stage in buffer cur (the order of tile_product's step)
  auto run = [&](int cur) {
    la.stage(cur ^ 1, some[cur ^ 1], tops[cur ^ 1], sA[cur ^ 1]);
    lb.stage(cur ^ 1, some[cur ^ 1], tops[cur ^ 1], sB[cur ^ 1]);
    fetch(cur ^ 1);
    frags(1, cur);
    __builtin_amdgcn_sched_barrier(0);
    multiply(0);
    __syncthreads();
    frags(0, cur ^ 1);
    __builtin_amdgcn_sched_barrier(0);
    multiply(1);
    const bool last = kinds & LAST;
    kinds >>= KIND;
    if (last) {
      store();
      cw = after(cw);
      clear();
    }
  };
  clear();
  open();
  fetch(0);
  ahead = 1;
  fetch(1);
  la.stage(0, some[0], tops[0], sA[0]);
  lb.stage(0, some[0], tops[0], sB[0]);
  ahead = 2;
  fetch(0);
  ahead = 3;
  __syncthreads();
  frags(0, 0);
  // (a stage past the last one ends no tile; leaving between the two would
  // make the waits at the top of the loop count that path's loads)
  do {
    run(0);
    run(1);
  } while (cw.at() < end);
}

// ---------------------------------------------------------------- float on BF16 matrix cores
// Float lists can also run as three-way BF16 splits: x = hi + mid + lo,
// hi = bf16(x), mid = bf16(x - hi), lo = bf16(x - hi - mid), each rounded
// to nearest even; the residuals are exact and lo takes the last 8 bits, so
// hi + mid + lo == x exactly for every normal float (down to ~2^-110,
// where lo would be subnormal).  BF16 keeps FP32's exponent range: no
// operand scaling, rows of any dynamic range.  Six
// v_mfma_f32_32x32x16_bf16 products per 16-deep k step (hl, lh, mm, hm, mh,
// hh: small terms first) with FP32 accumulation; the dropped ml, lm, ll
// terms are at most 2^-23 of |x y|.  An Inf or NaN enters as hi (mid = lo =
// 0), so non-finite values propagate as in FP32 arithmetic.  Each element
// is split once, when its k chunk is staged: LDS holds
// [stage][hi/mid/lo][row][32 k] as 16-byte segments, segment s of row r at
// s ^ ((r >> 1) & 3), so the 8 lanes of a 16-byte access hit distinct bank
// groups.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ uint32_t bf16_rne(uint32_t u) { return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16; }

__device__ __forceinline__ void split3_bf16(float x, uint32_t &h, uint32_t &m, uint32_t &l) {
  const uint32_t u = __float_as_uint(x);
  if ((u & 0x7f800000u) == 0x7f800000u) {                 // Inf keeps its bits, NaN becomes a quiet NaN
    h = (u & 0x7fffffu) ? (0x7fc0u | ((u >> 16) & 0x8000u)) : (u >> 16);
    m = 0;
    l = 0;
    return;
  }
  h = bf16_rne(u);
  if ((h & 0x7f80u) == 0x7f80u) h = u >> 16;             // above BF16's largest finite: truncate instead
  const float r = x - __uint_as_float(h << 16);            // exact
  m = bf16_rne(__float_as_uint(r));
  const float r2 = r - __uint_as_float(m << 16);           // exact
  l = bf16_rne(__float_as_uint(r2));                       // exact for normal x
}

constexpr int BKS = 32;   // k per chunk: two 16-deep MFMA steps

__device__ __forceinline__ void list_bf16x3_tile(const MmItem &it, int64_t tm, int64_t tn, uint4 (*As)[3][64][4],
                                                 uint4 (*Bs)[3][64][4]) {
  const float *a = (const float *)it.a + it.oa, *b = (const float *)it.b + it.ob;
  float *c = (float *)it.c;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, wr = w >> 1, wc = w & 1;
  const int H = (int)it.H, W = (int)it.W, K = (int)it.T;
  const int h0 = (int)tm * 64, w0 = (int)tn * 64;
  const int a_t = (int)it.a_t, a_h = (int)it.a_h, b_w = (int)it.b_w, b_t = (int)it.b_t;
  const bool active = h0 + 32 * wr < H && w0 + 32 * wc < W;
  // A: thread (row tid/4, 8 consecutive k of segment tid%4); B: thread
  // (column tid%64, 8 consecutive k of segment tid/64)
  const int arow = tid >> 2, aseg = tid & 3, bcol = tid & 63, bseg = tid >> 6;
  const int ah = h0 + arow < H ? h0 + arow : H - 1, bw = w0 + bcol < W ? w0 + bcol : W - 1;
  const bool avec = a_t == 1 && (((uintptr_t)(a + (int64_t)ah * a_h)) % 16 == 0);
  float ra[8], rb[8];
  auto load = [&](int k0) {
    const int ka = k0 + aseg * 8, kb = k0 + bseg * 8;
    if (avec && ka + 8 <= K) {
      const Vec<float, 4> x = *reinterpret_cast<const Vec<float, 4> *>(a + (int64_t)ah * a_h + ka);
      const Vec<float, 4> y = *reinterpret_cast<const Vec<float, 4> *>(a + (int64_t)ah * a_h + ka + 4);
#pragma unroll
      for (int e = 0; e < 4; e++) { ra[e] = x.v[e]; ra[4 + e] = y.v[e]; }
    } else {
#pragma unroll
      for (int e = 0; e < 8; e++) ra[e] = a[(int64_t)(ka + e < K ? ka + e : K - 1) * a_t + (int64_t)ah * a_h];
    }
#pragma unroll
    for (int e = 0; e < 8; e++) rb[e] = b[(int64_t)(kb + e < K ? kb + e : K - 1) * b_t + (int64_t)bw * b_w];
  };
  auto stage = [&](int buf, int k0) {
    uint32_t ph[4], pm[4], pl[4], qh[4], qm[4], ql[4];
    const bool arow_ok = h0 + arow < H, bcol_ok = w0 + bcol < W;
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      uint32_t h0_, m0_, l0_, h1_, m1_, l1_;
      const float x0 = (arow_ok && k0 + aseg * 8 + e < K) ? ra[e] : 0.0f;
      const float x1 = (arow_ok && k0 + aseg * 8 + e + 1 < K) ? ra[e + 1] : 0.0f;
      split3_bf16(x0, h0_, m0_, l0_);
      split3_bf16(x1, h1_, m1_, l1_);
      ph[e / 2] = h0_ | (h1_ << 16); pm[e / 2] = m0_ | (m1_ << 16); pl[e / 2] = l0_ | (l1_ << 16);
      const float y0 = (bcol_ok && k0 + bseg * 8 + e < K) ? rb[e] : 0.0f;
      const float y1 = (bcol_ok && k0 + bseg * 8 + e + 1 < K) ? rb[e + 1] : 0.0f;
      split3_bf16(y0, h0_, m0_, l0_);
      split3_bf16(y1, h1_, m1_, l1_);
      qh[e / 2] = h0_ | (h1_ << 16); qm[e / 2] = m0_ | (m1_ << 16); ql[e / 2] = l0_ | (l1_ << 16);
    }
    const int sa = aseg ^ ((arow >> 1) & 3), sb = bseg ^ ((bcol >> 1) & 3);
    As[buf][0][arow][sa] = make_uint4(ph[0], ph[1], ph[2], ph[3]);
    As[buf][1][arow][sa] = make_uint4(pm[0], pm[1], pm[2], pm[3]);
    As[buf][2][arow][sa] = make_uint4(pl[0], pl[1], pl[2], pl[3]);
    Bs[buf][0][bcol][sb] = make_uint4(qh[0], qh[1], qh[2], qh[3]);
    Bs[buf][1][bcol][sb] = make_uint4(qm[0], qm[1], qm[2], qm[3]);
    Bs[buf][2][bcol][sb] = make_uint4(ql[0], ql[1], ql[2], ql[3]);
  };
  lf32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; r++) acc[r] = 0.0f;
  if (K > 0) load(0);                  // an empty inner dimension loads nothing
  int buf = 0;
  const int fr = lane & 31, fseg = lane >> 5;
  const int ar_ = 32 * wr + fr, br_ = 32 * wc + fr;
  for (int k0 = 0; k0 < K; k0 += BKS) {
    stage(buf, k0);
    __syncthreads();
    if (k0 + BKS < K) load(k0 + BKS);
    {   // every wave multiplies (a branch here makes the
        // compiler copy the accumulators out of AGPRs and back each chunk)
#pragma unroll
      for (int ks = 0; ks < 2; ks++) {
        const int sa = (ks * 2 + fseg) ^ ((ar_ >> 1) & 3), sb = (ks * 2 + fseg) ^ ((br_ >> 1) & 3);
        bf16x8 fa[3], fb[3];
#pragma unroll
        for (int q = 0; q < 3; q++) {
          fa[q] = __builtin_bit_cast(bf16x8, As[buf][q][ar_][sa]);
          fb[q] = __builtin_bit_cast(bf16x8, Bs[buf][q][br_][sb]);
        }
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[0], fb[2], acc, 0, 0, 0);   // hi * lo
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[2], fb[0], acc, 0, 0, 0);   // lo * hi
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[1], fb[1], acc, 0, 0, 0);   // mid * mid
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[0], fb[1], acc, 0, 0, 0);   // hi * mid
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[1], fb[0], acc, 0, 0, 0);   // mid * hi
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[0], fb[0], acc, 0, 0, 0);   // hi * hi
      }
    }
    buf ^= 1;
  }
  if (active) {
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int64_t gh = h0 + 32 * wr + 8 * (r / 4) + 4 * (lane >> 5) + (r & 3);
      const int64_t gw = w0 + 32 * wc + (lane & 31);
      if (gh < H && gw < W) c[it.oc + gw * it.c_w + gh * it.c_h] = acc[r];
    }
  }
  __syncthreads();   // the LDS buffers are refilled by the next work item
}

__global__ __launch_bounds__(256) void list_bf16x3_queue(const MmItem *__restrict__ items,
                                                         const int3 *__restrict__ work,
                                                         const unsigned int *__restrict__ bounds,
                                                         unsigned int *counter) {
  __shared__ uint4 As[2][3][64][4];
  __shared__ uint4 Bs[2][3][64][4];
  __shared__ unsigned int next;
  int bin = blockIdx.x % LIST_BINS;
  unsigned done = 0;
  int3 job;
  while (list_next(counter, bounds, work, bin, done, &next, job)) list_bf16x3_tile(items[job.x], job.y, job.z, As, Bs);
}

__global__ __launch_bounds__(256) void list_bf16x3_one(const MmItem *__restrict__ items, int idx, int64_t ntn) {
  __shared__ uint4 As[2][3][64][4];
  __shared__ uint4 Bs[2][3][64][4];
  list_bf16x3_tile(items[idx], blockIdx.x / ntn, blockIdx.x % ntn, As, Bs);
}

static hipError_t list_bf16x3(const MmItem *d_items, const MmItem *h_items, int nitems, const int3 *d_work,
                              unsigned int *d_counter, bool each, int nblocks, hipStream_t s) {
  if (!each) {
    hipLaunchKernelGGL(list_reset, dim3(1), dim3(64), 0, s, d_counter);
    hipLaunchKernelGGL(list_bf16x3_queue, dim3(nblocks), dim3(256), 0, s, d_items, d_work,
                       (const unsigned int *)d_counter + LIST_BOUNDS, d_counter);
    return hipGetLastError();
  }
  for (int i = 0; i < nitems; i++) {
    const int64_t ntm = (h_items[i].H + 63) / 64, ntn = (h_items[i].W + 63) / 64;
    if (ntm * ntn == 0) continue;             // an empty k stores zeros
    hipLaunchKernelGGL(list_bf16x3_one, dim3((unsigned)(ntm * ntn)), dim3(256), 0, s, d_items, i, ntn);
  }
  return hipGetLastError();
}

template <class T> static int form_of(const MmItem &it) {
  if (it.T == 0) return 3;                // loads nothing of its operands
  const bool whole = it.T >= TILE_V<T>;   // as many k as one load takes
  return (it.a_t == 1 && whole ? 1 : 0) | (it.b_t == 1 && whole ? 2 : 0);
}
int list_form(int T, const MmItem &it) { return T == PDLHIP_D ? form_of<double>(it) : form_of<float>(it); }

template <class T, int TS>
static hipError_t list_tiles_T(const MmItem *d_items, const MmItem *h_items, int nitems, const ListPart *parts,
                               int nparts, bool each, hipStream_t s) {
  auto go = [&](int form, unsigned grid, const int3 *work, const unsigned int *bounds, int only, unsigned ntn) {
    if (form == 3)
      hipLaunchKernelGGL((list_tiles<T, TS, true, true>), dim3(grid), dim3(256), 0, s, d_items, work, bounds, only, ntn);
    else if (form == 1)
      hipLaunchKernelGGL((list_tiles<T, TS, true, false>), dim3(grid), dim3(256), 0, s, d_items, work, bounds, only, ntn);
    else if (form == 2)
      hipLaunchKernelGGL((list_tiles<T, TS, false, true>), dim3(grid), dim3(256), 0, s, d_items, work, bounds, only, ntn);
    else
      hipLaunchKernelGGL((list_tiles<T, TS, false, false>), dim3(grid), dim3(256), 0, s, d_items, work, bounds, only, ntn);
  };
  if (!each) {   // as many blocks as are resident at once
    for (int i = 0; i < nparts; i++)
      go(parts[i].form, LIST_BINS * std::min(std::max(parts[i].longest, 1u), 32u * LIST_PER_CU<TS>), parts[i].work,
         parts[i].bounds, 0, 1);
    return hipGetLastError();
  }
  for (int i = 0; i < nitems; i++) {
    const int64_t ntm = (h_items[i].H + TS - 1) / TS, ntn = (h_items[i].W + TS - 1) / TS;
    if (ntm * ntn == 0) continue;             // an empty k stores zeros
    go(form_of<T>(h_items[i]), (unsigned)(ntm * ntn), nullptr, nullptr, i, (unsigned)ntn);
  }
  return hipGetLastError();
}

template <class T>
static hipError_t list_T(const MmItem *d_items, const MmItem *h_items, int nitems, const int3 *d_work,
                         unsigned int *d_counter, int tile, bool fused, bool each, int nblocks, hipStream_t s) {
#define LQ(F, TS) hipLaunchKernelGGL((list_queue<T, F, TS>), dim3(nblocks), dim3(256), 0, s, d_items, d_work, \
                                     (const unsigned int *)d_counter + LIST_BOUNDS + (TS == 32 ? LIST_BINS + 1 : 0), \
                                     d_counter)
#define L1(F, TS) hipLaunchKernelGGL((list_one<T, F, TS>), dim3((unsigned)(ntm * ntn)), dim3(256), 0, s, d_items, i, ntn)
  if (!each) {
    hipLaunchKernelGGL(list_reset, dim3(1), dim3(64), 0, s, d_counter);
    if (tile == 32) { if (fused) LQ(true, 32); else LQ(false, 32); }
    else { if (fused) LQ(true, 64); else LQ(false, 64); }
    return hipGetLastError();
  }
  for (int i = 0; i < nitems; i++) {
    const int64_t ntm = (h_items[i].H + tile - 1) / tile, ntn = (h_items[i].W + tile - 1) / tile;
    if (ntm * ntn == 0) continue;
    if (tile == 32) { if (fused) L1(true, 32); else L1(false, 32); }
    else { if (fused) L1(true, 64); else L1(false, 64); }
  }
#undef LQ
#undef L1
  return hipGetLastError();
}

hipError_t launch_matmult_list(int T, const MmItem *d_items, const MmItem *h_items, int nitems, const int3 *d_work,
                               unsigned int *d_counter, const ListPart *parts, int nparts, int tile, bool fused,
                               bool each, int nblocks, hipStream_t s) {
  // tile 0 / 2: the matrix-core kernels (64x64 / 32x32 work items), float and
  // double lists in the default modes; tile 1: float on the BF16 matrix cores
  if (tile == 1 && fused && T == PDLHIP_F)
    return list_bf16x3(d_items, h_items, nitems, d_work, d_counter, each, nblocks, s);
  if (tile == 1) tile = 0;
  if (fused && T == PDLHIP_F && (tile == 0 || tile == 2))
    return tile == 0 ? list_tiles_T<float, 64>(d_items, h_items, nitems, parts, nparts, each, s)
                     : list_tiles_T<float, 32>(d_items, h_items, nitems, parts, nparts, each, s);
  if (fused && T == PDLHIP_D && (tile == 0 || tile == 2))
    return tile == 0 ? list_tiles_T<double, 64>(d_items, h_items, nitems, parts, nparts, each, s)
                     : list_tiles_T<double, 32>(d_items, h_items, nitems, parts, nparts, each, s);
  if (tile == 0) tile = 64;
  if (tile == 2) tile = 32;
  switch (T) {
#define X(TC) case TC: return list_T<CType<TC>::T>(d_items, h_items, nitems, d_work, d_counter, tile, fused, each, \
                                                   nblocks, s);
    PDLHIP_FOR_EACH_TYPE(X)
#undef X
  default: return hipErrorInvalidValue;
  }
}

}  // namespace pdlhip
