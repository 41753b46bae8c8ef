// The C tile of a float or double product on the FP32 / FP64 matrix cores,
// shared by the single and batched products (k_tile.hip) and the matmult
// lists (k_batch.hip): products and sums in the operands' own type.
//
// v_mfma_f64_16x16x4_f64 and v_mfma_f32_16x16x4_f32: lane l holds A[l%16][k]
// and B[k][l%16] for its k = l / 16 of four; result register r of lane l is
// D[4r + l/16][l%16] (double) or D[4 (l/16) + r][l%16] (float).
//
// A block of 4 waves computes BM x BN of C.  Operands go global -> registers
// -> LDS in stages of 128 bytes of k (16 doubles, 32 floats), two stages'
// loads in flight while the matrix cores work on a third.  LDS rows hold a
// stage, padded by 16 bytes: a lane reads 16 bytes of neighbouring k of its
// row (eight rows fall on distinct bank groups) and feeds them to two (four)
// instructions; which k an instruction covers is free as long as A and B
// agree.
#pragma once

#include <hip/hip_runtime.h>

#include "device.hpp"

namespace pdlhip {

template <class T> struct TileType;
template <> struct TileType<double> {
  typedef double acc_t __attribute__((ext_vector_type(4)));
  typedef double vec_t __attribute__((ext_vector_type(2)));
  __device__ static __forceinline__ acc_t mfma(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  __device__ static __forceinline__ int row(int r, int q) { return 4 * r + q; }
};
template <> struct TileType<float> {
  typedef float acc_t __attribute__((ext_vector_type(4)));
  typedef float vec_t __attribute__((ext_vector_type(4)));
  __device__ static __forceinline__ acc_t mfma(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  __device__ static __forceinline__ int row(int r, int q) { return 4 * q + r; }
};
template <class T> constexpr int TILE_K = 128 / (int)sizeof(T);              // k of a stage
template <class T> constexpr int TILE_V = 16 / (int)sizeof(T);               // k of a 16-byte access
template <class T> constexpr int TILE_P = TILE_K<T> + TILE_V<T>;              // an LDS row

// One operand's share of a stage: N rows x 8 groups of 16 bytes of k over 256
// threads.  KFAST (unit stride along k): neighbouring threads take
// neighbouring groups, one load each (which the hardware takes at any
// element's address); else neighbouring threads take neighbouring rows.  The
// first stage takes the k that do not fill a stage (or a whole one), so that
// the loop's loads are whole, sit behind no branch, and their waits are
// counted.
template <class T, int N, bool KFAST> struct TileLoad {
  static constexpr int P = N * 8 / 256, V = TILE_V<T>;
  typedef typename TileType<T>::vec_t vec;
  typedef vec __attribute__((aligned(sizeof(T)))) vecu;
  gptr<const T> ptr[P];   // (stated global: a generic pointer would load through the flat path)
  vec v[2][P];            // two stages on their way
  __device__ static int row(int s) { const int e = threadIdx.x + 256 * s; return KFAST ? e / 8 : e % N; }
  __device__ static int group(int s) { const int e = threadIdx.x + 256 * s; return KFAST ? e % 8 : e / N; }
  // the first stage's `some` k, zeros after them, into l; rows past the
  // operand's last repeat it: they reach only outputs that are not stored
  __device__ void first(const T *base, int64_t r0, int64_t R, int64_t inc_r, int64_t k0, int64_t inc_k, int some,
                        T (*l)[TILE_P<T>]) {
#pragma unroll
    for (int s = 0; s < P; s++) {
      const int64_t r = r0 + row(s) < R ? r0 + row(s) : R - 1;
      ptr[s] = as_global(base + r * inc_r + (k0 + V * group(s)) * inc_k);
    }
    if (some == TILE_K<T>) {
      load(0, inc_k, false);
    } else {
#pragma unroll
      for (int s = 0; s < P; s++)
#pragma unroll
        for (int i = 0; i < V; i++) v[0][s][i] = V * group(s) + i < some ? ptr[s][i * inc_k] : T(0);
    }
    stage(0, l);
#pragma unroll
    for (int s = 0; s < P; s++) ptr[s] += some * inc_k;
  }
  // the stage at ptr, which moves on if another follows
  __device__ void load(int set, int64_t inc_k, bool more) {
#pragma unroll
    for (int s = 0; s < P; s++) {
      if (KFAST) v[set][s] = *(gptr<const vecu>)ptr[s];
      else
#pragma unroll
        for (int i = 0; i < V; i++) v[set][s][i] = ptr[s][i * inc_k];
    }
    const int64_t step = more ? TILE_K<T> * inc_k : 0;
#pragma unroll
    for (int s = 0; s < P; s++) ptr[s] += step;
  }
  __device__ void stage(int set, T (*l)[TILE_P<T>]) {
#pragma unroll
    for (int s = 0; s < P; s++) *reinterpret_cast<vec *>(&l[row(s)][V * group(s)]) = v[set][s];
  }
};

// how a tile sums: a stage's k at a time (double: one chain), 8 k at a time
// (float), or 8 k at a time where all of k is half a stage or less
constexpr int BY_STAGE = 0, BY_EIGHT = 1, HALF_STAGE = 2;
template <int HOW> constexpr int TILE_BUFS = HOW == HALF_STAGE ? 1 : 2;   // stages in LDS

// the tile at (m0, n0) summed over k in [kb, ke), ke > kb; put(row, column,
// value) for each of the thread's outputs, counted within the tile
template <class T, int BM, int BN, int WR, int WC, bool AK, bool BK, int HOW, class Put>
__device__ __forceinline__ void tile_product(const T *a, const T *b, int64_t H, int64_t W, int64_t a_h, int64_t a_t,
                                             int64_t b_w, int64_t b_t, int64_t m0, int64_t n0, int64_t kb, int64_t ke,
                                             T (*sA)[BM][TILE_P<T>], T (*sB)[BN][TILE_P<T>], Put put) {
  constexpr int TI = BM / WR / 16, TJ = BN / WC / 16, KB = TILE_K<T>, V = TILE_V<T>;
  static_assert(WR * WC == 4, "four waves");
  typedef TileType<T> TT;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wr = w / WC, wc = w % WC, fr = lane & 15, fk = lane >> 4;
  TileLoad<T, BM, AK> la;
  TileLoad<T, BN, BK> lb;
  typename TT::acc_t acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; i++)
#pragma unroll
    for (int j = 0; j < TJ; j++) acc[i][j] = typename TT::acc_t{T(0), T(0), T(0), T(0)};
  const int some = (int)((ke - kb - 1) % KB) + 1;
  const int64_t n = (ke - kb - some) / KB + 1;   // stages
  la.first(a, m0, H, a_h, kb, a_t, some, sA[0]);
  lb.first(b, n0, W, b_w, kb, b_t, some, sB[0]);
  // A step multiplies the two halves of a stage.  The barrier stands between
  // them: before it the next stage goes to the other buffer (whose last
  // reads came before the barrier of the step before) and the second half's
  // fragments are read, after it the next step's first half, so that every
  // LDS read has a half's matrix instructions to arrive in.
  auto fetch = [&](int set, int64_t q) {   // stage q (past the last one, that again, unused)
    la.load(set, a_t, q + 1 < n);
    lb.load(set, b_t, q + 1 < n);
  };
  typename TT::vec_t af[2][TI], bf[2][TJ];
  auto frags = [&](int half, int buf) {
#pragma unroll
    for (int i = 0; i < TI; i++)
      af[half][i] = *reinterpret_cast<const typename TT::vec_t *>(&sA[buf][(wr * TI + i) * 16 + fr][half * KB / 2 + V * fk]);
#pragma unroll
    for (int j = 0; j < TJ; j++)
      bf[half][j] = *reinterpret_cast<const typename TT::vec_t *>(&sB[buf][(wc * TJ + j) * 16 + fr][half * KB / 2 + V * fk]);
  };
  // Double: one chain of sums per output.  Float: the matrix cores round at
  // every k, so a few k at a time are summed from zero and their sum added to
  // the total: a stage's 32 k, or 8 where there are few.  The error of
  // 1024^3 is then 1.5e-7 instead of 5.7e-7, of 64^3 8e-8 instead of 1.5e-7
  // (the FP16 split's: 3.5e-7 and 9e-8); the adds run on the vector unit
  // while the matrix cores go on with the other tiles.
  typename TT::acc_t part[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; i++)
#pragma unroll
    for (int j = 0; j < TJ; j++) part[i][j] = acc[i][j];
  auto multiply = [&](int half) {
#pragma unroll
    for (int u = 0; u < V; u++)
#pragma unroll
      for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++) {
          if constexpr (sizeof(T) == 8) {
            acc[i][j] = TT::mfma(af[half][i][u], bf[half][j][u], acc[i][j]);
          } else {
            const bool fresh = HOW != BY_STAGE ? u % 2 == 0 : half == 0 && u == 0;
            if (fresh) acc[i][j] += part[i][j];
            part[i][j] = TT::mfma(af[half][i][u], bf[half][j][u], fresh ? typename TT::acc_t{} : part[i][j]);
          }
        }
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
  if (HOW != HALF_STAGE && n > 1) {
    fetch(1, 1);
    fetch(0, 2);
  }
  __syncthreads();
  frags(0, 0);
  if constexpr (HOW == HALF_STAGE) {
    multiply(0);
  } else {
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
  }
  if constexpr (sizeof(T) == 4) {
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
      for (int j = 0; j < TJ; j++) acc[i][j] += part[i][j];
  }
#pragma unroll
  for (int i = 0; i < TI; i++)
#pragma unroll
    for (int j = 0; j < TJ; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) put((wr * TI + i) * 16 + TT::row(r, fk), (wc * TJ + j) * 16 + fr, acc[i][j][r]);
}

}  // namespace pdlhip
