// Reductions and scans of lib/PDL/Ufunc.pd over the core dim n (dim 0 of a),
// one output element per broadcast position:
//   sumover/prodover (+d)       Ufunc.pd:88-118
//   cumusumover/cumuprodover    Ufunc.pd:120-140
//   average/daverage            Ufunc.pd:413-444
//   minimum/maximum(+_ind)      Ufunc.pd:446-482
//   minimum_n_ind/maximum_n_ind Ufunc.pd:484-540
//   minmaximum                  Ufunc.pd:563-613
//
// Kernels:
//   wave   1, 4 or 16 wavefronts per output (rows with unit stride), 16-byte
//          vector loads, cross-lane combine with shuffles.
//   split  the longest rows and few outputs: blocks reduce row chunks into partials
//          in scratch, a second kernel combines them.
//   grid   strided rows and rows shorter than a wave: a block's threads cover
//          outputs x positions along n, n cut into chunks where the outputs
//          alone leave the chip idle (partials combined as for split).
//   scan   integer scans of unit-stride rows: blocks scan chunks through LDS.
//   seq    scans in PDL's order: a lane per row in LDS, other waves moving.
//   thread one thread per output walking n in index order (float products,
//          *_n_ind, the shortest rows and columns): adjacent threads read
//          adjacent addresses when the broadcast dim 0 is the contiguous one.
//
// Semantics kept exactly: integer sums/products wrap in the output type
// (any order gives PDL's bits), min/max follow PDL's rules (a NaN never
// displaces a non-NaN, a non-NaN displaces a NaN, ties keep the first,
// all-NaN gives the last), bad values are skipped, empty/all-bad rows give
// BAD (or 0 / NaN for average in good mode).  Float sums are compensated
// (Neumaier per lane, double-double across lanes and blocks), so they are
// at least as accurate as PDL's sequential float loop; float products and
// float scans run in PDL's exact sequential order.
#include <hip/hip_runtime.h>

#include "device.hpp"
#include "launch.hpp"
#include "reduce_common.hpp"

namespace pdlhip {

void *scratch_alloc(size_t bytes);
void scratch_free(void *p);
void *partials_alloc(size_t bytes);
void partials_free(void *p);

__device__ inline void out_offsets(const RedPlan &p, int64_t e, int64_t *off) {
  for (int k = 0; k < p.npdl; k++) off[k] = p.off[k];
  for (int d = 0; d < p.nd; d++) {
    int64_t i = e % p.dims[d];
    e /= p.dims[d];
    for (int k = 0; k < p.npdl; k++) off[k] += i * p.inc[k][d];
  }
}

// ---------------------------------------------------------------- rows
constexpr int RT = 256;  // threads per block (4 waves)

// lane of NL cooperating lanes takes its share of elements [begin, end) of a
// unit-stride row: the elements up to the first 16-byte boundary one to a
// lane, then 16-byte vectors, then the rest one to a lane, each lane's in
// increasing index order.  (Rows of odd length start unaligned; loading those
// an element at a time took 167 us for 64 rows of 32091 ints.)
// ON16: every row starts on such a boundary, and a short one is spared the
// search for it (1000000 rows of 64 floats: 346 us, 372 with it).
template <int OP, class Tin, class Tacc, bool BAD, int NL, bool ON16 = false>
__device__ inline void row_segment(Part<Tin, Tacc> &pt, const Tin *__restrict__ row, int64_t begin, int64_t end,
                                   int lane, const BadInfo &ba, bool stream) {
  constexpr int VEC = 16 / sizeof(Tin);
  // 16-byte loads in flight per lane: 4 for 4- and 8-byte elements, 2 for
  // the narrower ones (eight or sixteen elements per load already)
  constexpr int RED_U = sizeof(Tin) >= 4 ? 4 : 2;
  const Tin abv = bv_as<Tin>(ba.bv);
  const int64_t lead = ON16 ? 0 : ((16 - (int)((uintptr_t)(row + begin) & 15)) & 15) / sizeof(Tin);
  const int64_t vb = begin + lead < end ? begin + lead : end, ve = vb + (end - vb) / VEC * VEC;
  // only floats have NaN for a bad value: without its test an element's mask is
  // one compare (1000000 rows of 64 bytes with bad values: 273 us, 335 with it)
  const int nan = IsFloat<Tin>::v ? ba.isnan : 0;
  auto push = [&](Tin x, int64_t i) {
    if constexpr (BAD) { if (isbad(x, abv, nan)) return; }
    part_push<OP, Tin, Tacc>(pt, x, i);
  };
  if (!ON16 && begin + lane < vb) push(row[begin + lane], begin + lane);
  int64_t i = vb + (int64_t)lane * VEC;
  for (; i + (RED_U - 1) * NL * VEC < ve; i += RED_U * NL * VEC) {
    Vec<Tin, VEC> x[RED_U];
#pragma unroll
    for (int u = 0; u < RED_U; u++)
      x[u] = stream ? load_nt<Tin, VEC>(row + i + u * NL * VEC)
                    : *reinterpret_cast<const Vec<Tin, VEC> *>(row + i + u * NL * VEC);
#pragma unroll
    for (int u = 0; u < RED_U; u++)
#pragma unroll
      for (int k = 0; k < VEC; k++) push(x[u].v[k], i + u * NL * VEC + k);
  }
  for (; i < ve; i += NL * VEC) {
    const Vec<Tin, VEC> x = stream ? load_nt<Tin, VEC>(row + i) : *reinterpret_cast<const Vec<Tin, VEC> *>(row + i);
#pragma unroll
    for (int k = 0; k < VEC; k++) push(x.v[k], i + k);
  }
  if (ve + lane < end) push(row[ve + lane], ve + lane);
}

// the NW waves of a block join their partials (each already combined within
// the wave); the result is in thread 0
template <int OP, class Tin, class Tacc, int NW>
__device__ inline void waves_join(Part<Tin, Tacc> &pt, Part<Tin, Tacc> *sh) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) sh[w] = pt;
  __syncthreads();
  if (w == 0) {
    part_init<OP, Tin, Tacc>(pt);
    if (lane < NW) pt = sh[lane];
    wave_reduce<OP, Tin, Tacc>(pt);
  }
}

// NW waves per row; four rows per block of 256 threads for NW = 1, else a
// row per block
template <int OP, class Tin, class Tout, class Tacc, bool BAD, int NW, bool ON16 = false>
__global__ __launch_bounds__(NW > 4 ? NW * 64 : RT) void red_wave(const Tin *__restrict__ a, RedPlan p, Outs o,
                                                                  BadInfo ba, bool stream) {
  constexpr int PER = NW == 1 ? 4 : 1;
  __shared__ Part<Tin, Tacc> sh[NW];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int64_t e = (int64_t)blockIdx.x * PER + (NW == 1 ? w : 0); e < p.nout; e += (int64_t)gridDim.x * PER) {
    int64_t off[MAXP];
    out_offsets(p, e, off);
    Part<Tin, Tacc> pt;
    part_init<OP, Tin, Tacc>(pt);
    row_segment<OP, Tin, Tacc, BAD, NW * 64, ON16>(pt, a + off[0], 0, p.n, NW == 1 ? lane : (int)threadIdx.x, ba, stream);
    wave_reduce<OP, Tin, Tacc>(pt);
    if constexpr (NW > 1) {
      waves_join<OP, Tin, Tacc, NW>(pt, sh);
      if (threadIdx.x == 0) part_store<OP, Tin, Tout, Tacc>(pt, o, off, BAD);
      __syncthreads();   // sh is refilled for the next row
    } else {
      if (lane == 0) part_store<OP, Tin, Tout, Tacc>(pt, o, off, BAD);
    }
  }
}

// ---------------------------------------------------------------- split
// stage 1: block (e, k) reduces chunk k of row e into parts[e * nchunk + k]
template <int OP, class Tin, class Tout, class Tacc, bool BAD>
__global__ __launch_bounds__(RT) void red_split1(const Tin *__restrict__ a, RedPlan p, int64_t nchunk, int64_t clen,
                                                 Part<Tin, Tacc> *parts, BadInfo ba, bool stream) {
  __shared__ Part<Tin, Tacc> sh[RT / 64];
  const int64_t e = blockIdx.x / nchunk, k = blockIdx.x % nchunk;
  int64_t off[MAXP];
  out_offsets(p, e, off);
  const int64_t cb = k * clen, ce = (cb + clen < p.n) ? cb + clen : p.n;
  Part<Tin, Tacc> pt;
  part_init<OP, Tin, Tacc>(pt);
  row_segment<OP, Tin, Tacc, BAD, RT>(pt, a + off[0], cb, ce, threadIdx.x, ba, stream);
  wave_reduce<OP, Tin, Tacc>(pt);
  waves_join<OP, Tin, Tacc, RT / 64>(pt, sh);
  if (threadIdx.x == 0) parts[blockIdx.x] = pt;
}

// the R partials of each output, `step` apart in sh, meet in a tree; the
// result is in the thread with r == 0
template <int OP, class Tin, class Tacc>
__device__ inline void block_tree(Part<Tin, Tacc> &pt, Part<Tin, Tacc> *sh, bool in, int r, int R, int step) {
  sh[threadIdx.x] = pt;
  for (int h = R > 1 ? 1 << (31 - __builtin_clz(R - 1)) : 0; h >= 1; h >>= 1) {
    __syncthreads();
    if (in && r < h && r + h < R) {
      part_combine<OP>(pt, sh[threadIdx.x + h * step]);
      sh[threadIdx.x] = pt;
    }
  }
}

// stage 2: G threads (a power of two, about four chunks each) combine the
// partials of one row.  A wave per row walked 2048 chunks 32 to a lane, one
// dependent load after another, and made half of a column sum (41 us, now 25).
template <int OP, class Tin, class Tout, class Tacc, bool BAD>
__global__ __launch_bounds__(RT) void red_split2(RedPlan p, int64_t nchunk, int G, const Part<Tin, Tacc> *parts,
                                                 Outs o) {
  __shared__ Part<Tin, Tacc> sh[RT];
  const int r = threadIdx.x % G;
  const int64_t e = (int64_t)blockIdx.x * (RT / G) + threadIdx.x / G;
  const bool in = e < p.nout;
  Part<Tin, Tacc> pt;
  part_init<OP, Tin, Tacc>(pt);
  if (in) {
#pragma unroll 4
    for (int64_t k = r; k < nchunk; k += G) part_combine<OP>(pt, parts[e * nchunk + k]);
  }
  block_tree<OP>(pt, sh, in, r, G, 1);
  if (in && r == 0) {
    int64_t off[MAXP];
    out_offsets(p, e, off);
    part_store<OP, Tin, Tout, Tacc>(pt, o, off, BAD);
  }
}

template <int OP, class Tin, class Tout, class Tacc, bool BAD>
static void split2_launch(const RedPlan &p, int64_t nchunk, const Part<Tin, Tacc> *parts, const Outs &o,
                          hipStream_t s) {
  int G = 1;
  while (G < RT && G * 4 < nchunk) G *= 2;
  const int64_t per = RT / G;
  hipLaunchKernelGGL((red_split2<OP, Tin, Tout, Tacc, BAD>), dim3((unsigned)((p.nout + per - 1) / per)), dim3(RT), 0, s,
                     p, nchunk, G, parts, o);
}

// ---------------------------------------------------------------- grid
// A block covers LE outputs x R positions along n (LE * R <= 256 threads):
// thread (e, r) takes elements r, r + R, ... of its chunk of row e, eight
// loads in flight, then the R partials of an output meet in a tree in LDS.
// NFAST puts n on neighbouring threads (rows whose stride along n is the
// smaller one, such as short unit-stride rows and stepped slices), otherwise
// outputs are neighbours (columns of a table), so that a wave reads
// neighbouring addresses either way.  Bound by HBM; one thread per output
// walking n took 187 ms (0.5 GB/s) to average 24 columns of 1000003 floats,
// this takes 25 us with the combine (19.3 + 5.4, 4.9 TB/s in this kernel).
constexpr int GRID_U = 8;
template <int OP, class Tin, class Tout, class Tacc, bool BAD, bool NFAST>
__global__ __launch_bounds__(RT) void red_grid(const Tin *__restrict__ a, RedPlan p, Outs o, BadInfo ba, int LE, int R,
                                               int64_t nchunk, int64_t clen, Part<Tin, Tacc> *parts) {
  __shared__ Part<Tin, Tacc> sh[RT];
  const Tin abv = bv_as<Tin>(ba.bv);
  const int r = NFAST ? threadIdx.x % R : threadIdx.x / LE, el = NFAST ? threadIdx.x / R : threadIdx.x % LE;
  const int64_t k = blockIdx.x % nchunk;
  const int64_t cb = k * clen, ce = (cb + clen < p.n) ? cb + clen : p.n;
  const int64_t ngroup = (p.nout + LE - 1) / LE;
  for (int64_t gr = blockIdx.x / nchunk; gr < ngroup; gr += gridDim.x / nchunk) {
    const int64_t e = gr * LE + el;
    const bool in = e < p.nout && r < R && el < LE;
    int64_t off[MAXP];
    Part<Tin, Tacc> pt;
    part_init<OP, Tin, Tacc>(pt);
    if (in) {
      out_offsets(p, e, off);
      const Tin *ap = a + off[0];
      const int64_t inc = p.inc_n[0];
      int64_t i = cb + r;
      for (; i + (int64_t)(GRID_U - 1) * R < ce; i += (int64_t)GRID_U * R) {
        Tin x[GRID_U];
#pragma unroll
        for (int u = 0; u < GRID_U; u++) x[u] = ap[(i + (int64_t)u * R) * inc];
#pragma unroll
        for (int u = 0; u < GRID_U; u++) {
          if constexpr (BAD) { if (isbad(x[u], abv, ba.isnan)) continue; }
          part_push<OP, Tin, Tacc>(pt, x[u], i + (int64_t)u * R);
        }
      }
      // the rest, fewer than GRID_U of them: loaded together as well
      Tin x[GRID_U];
#pragma unroll
      for (int u = 0; u < GRID_U - 1; u++) {
        const int64_t q = i + (int64_t)u * R;
        x[u] = q < ce ? ap[q * inc] : Tin(0);
      }
#pragma unroll
      for (int u = 0; u < GRID_U - 1; u++) {
        const int64_t q = i + (int64_t)u * R;
        if (q >= ce) continue;
        if constexpr (BAD) { if (isbad(x[u], abv, ba.isnan)) continue; }
        part_push<OP, Tin, Tacc>(pt, x[u], q);
      }
    }
    if (R > 1) block_tree<OP>(pt, sh, in, r, R, NFAST ? 1 : LE);
    if (in && r == 0) {
      if (nchunk == 1) part_store<OP, Tin, Tout, Tacc>(pt, o, off, BAD);
      else parts[e * nchunk + k] = pt;
    }
    if (R > 1) __syncthreads();   // sh is refilled for the next group
  }
}

// ---------------------------------------------------------------- scan
// Integer cumusumover/cumuprodover with unit-stride rows: one block per row,
// chunks of 4096 staged through LDS (coalesced in and out), a sequential scan
// of 16 elements per thread, then wave and block prefix combines.  Wrapping
// integer + and * are associative, so the result has PDL's exact bits.  A bad
// element contributes the identity and is written as the output's bad value
// (Ufunc.pd:127-132).  Few long rows are cut into chunks of a multiple of 4096
// elements, a block each: scan_totals leaves every chunk's total, and a
// chunk's scan starts from the totals before it (16 rows of 1000000 ints:
// 520 us with a block per row, 13 + 24 with chunks).  Whole rows (not CUT) are
// a form of their own (4096 of 1000 ints: 15 us, 16 with the chunk's tests).
constexpr int SC_IT = 16, SC_CH = RT * SC_IT;
__device__ inline int sc_pad(int i) { return i + (i >> 4); }

template <int OP, class Tin, class Tout, bool BAD>
__global__ __launch_bounds__(RT) void scan_totals(const Tin *__restrict__ a, RedPlan p, BadInfo ba, int64_t nchunk,
                                                  int64_t clen, Tout *totals) {
  constexpr int ROP = OP == R_CUMUPROD ? R_PROD : R_SUM;
  __shared__ Part<Tin, Tout> sh[RT / 64];
  const int64_t e = blockIdx.x / nchunk, k = blockIdx.x % nchunk;
  int64_t off[MAXP];
  out_offsets(p, e, off);
  const int64_t cb = k * clen, ce = cb + clen < p.n ? cb + clen : p.n;
  Part<Tin, Tout> pt;
  part_init<ROP, Tin, Tout>(pt);
  row_segment<ROP, Tin, Tout, BAD, RT>(pt, a + off[0], cb, ce, threadIdx.x, ba, false);
  wave_reduce<ROP, Tin, Tout>(pt);
  waves_join<ROP, Tin, Tout, RT / 64>(pt, sh);
  if (threadIdx.x == 0) totals[blockIdx.x] = pt.s;
}

template <int OP, class Tin, class Tout, bool BAD, bool CUT>
__global__ __launch_bounds__(RT) void scan_rows(const Tin *__restrict__ a, RedPlan p, Outs o, BadInfo ba, int64_t nchunk,
                                                int64_t clen, const Tout *totals) {
  constexpr bool PR = (OP == R_CUMUPROD);
  __shared__ Tout sh[SC_CH + SC_CH / 16];
  __shared__ uint8_t badm[BAD ? SC_CH : 1];
  __shared__ Tout wsum[RT / 64];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const Tin abv = bv_as<Tin>(ba.bv);
  const Tout obv = bv_as<Tout>(o.bv[0]);
  const Tout ident = PR ? Tout(1) : Tout(0);
  for (int64_t q = blockIdx.x; q < (CUT ? p.nout * nchunk : p.nout); q += gridDim.x) {
    const int64_t e = CUT ? q / nchunk : q, k = CUT ? q - e * nchunk : 0;
    int64_t off[MAXP];
    out_offsets(p, e, off);
    const Tin *ap = a + off[0];
    Tout *bp = (Tout *)o.p[0] + off[1];
    Tout carry = ident;
    if (CUT && k > 0) {   // the totals of the row's chunks before this one
      Tout t = ident;
      for (int64_t i = tid; i < k; i += RT) t = PR ? wmul(t, totals[e * nchunk + i]) : wadd(t, totals[e * nchunk + i]);
#pragma unroll
      for (int m = 32; m >= 1; m >>= 1) {
        const Tout u = shfl_xor(t, m);
        t = PR ? wmul(t, u) : wadd(t, u);
      }
      if (lane == 0) wsum[w] = t;
      __syncthreads();
#pragma unroll
      for (int i = 0; i < RT / 64; i++) carry = PR ? wmul(carry, wsum[i]) : wadd(carry, wsum[i]);
      __syncthreads();
    }
    const int64_t end = CUT && (k + 1) * clen < p.n ? (k + 1) * clen : p.n;
    for (int64_t c0 = CUT ? k * clen : 0; c0 < end; c0 += SC_CH) {
      const int len = (end - c0 < SC_CH) ? (int)(end - c0) : SC_CH;
      // every load of the chunk is issued before the first LDS write
      Tin xv[SC_IT];
#pragma unroll
      for (int k = 0; k < SC_IT; k++) {
        const int idx = tid + RT * k;
        xv[k] = idx < len ? ap[c0 + idx] : Tin(0);
      }
#pragma unroll
      for (int k = 0; k < SC_IT; k++) {
        const int idx = tid + RT * k;
        Tout v = ident;
        if (idx < len) {
          bool isb = false;
          if constexpr (BAD) { isb = isbad(xv[k], abv, ba.isnan); badm[idx] = isb; }
          if (!isb) v = (Tout)xv[k];
        }
        sh[sc_pad(idx)] = v;
      }
      __syncthreads();
      // sequential scan of this thread's 16 consecutive elements
      Tout run = ident;
      const int base = tid * SC_IT;
#pragma unroll
      for (int j = 0; j < SC_IT; j++) {
        run = PR ? wmul(run, sh[sc_pad(base + j)]) : wadd(run, sh[sc_pad(base + j)]);
        sh[sc_pad(base + j)] = run;
      }
      // inclusive wave scan of the thread totals
      Tout incl = run;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        Tout t = shfl_up(incl, d);
        if (lane >= d) incl = PR ? wmul(t, incl) : wadd(t, incl);
      }
      Tout excl = shfl_up(incl, 1);
      if (lane == 0) excl = ident;
      if (lane == 63) wsum[w] = incl;
      __syncthreads();
      Tout wpre = ident, tot = ident;
#pragma unroll
      for (int k = 0; k < RT / 64; k++) {
        if (k < w) wpre = PR ? wmul(wpre, wsum[k]) : wadd(wpre, wsum[k]);
        tot = PR ? wmul(tot, wsum[k]) : wadd(tot, wsum[k]);
      }
      Tout pre = PR ? wmul(wmul(carry, wpre), excl) : wadd(wadd(carry, wpre), excl);
#pragma unroll
      for (int j = 0; j < SC_IT; j++) {
        Tout v = sh[sc_pad(base + j)];
        sh[sc_pad(base + j)] = PR ? wmul(pre, v) : wadd(pre, v);
      }
      __syncthreads();
#pragma unroll
      for (int k = 0; k < SC_IT; k++) {
        const int idx = tid + RT * k;
        if (idx < len) {
          Tout v = sh[sc_pad(idx)];
          if constexpr (BAD) { if (badm[idx]) v = obv; }
          bp[c0 + idx] = v;
        }
      }
      carry = PR ? wmul(carry, tot) : wadd(carry, tot);
      __syncthreads();
    }
  }
}

// Scans in PDL's own order, element after element (float and double sums and
// products, whose rounding that order defines; Ufunc.pd:120-140), and scans
// of short or strided rows of any type.  The chain of one row is serial, so
// this is bound by it until there are rows enough to be bound by HBM.  In a
// block three waves bring in the next chunk of C elements of each of G rows
// and store the one before (along whichever of n and rows is the closer in
// memory) while the first wave scans:
//   G > 1   a lane per row, out of LDS and back, 16 bytes at a time
//   one row the lanes hold the chunk in registers, K neighbours each, and add
//           in turn, so that the chain has no LDS access in it (9 cycles
//           per element against 15.4 through LDS)
// One thread per row straight from memory took 52.4 ms for a row of 476006
// floats, this takes 1.8 ms; 60000 rows of 256: 27 us (4.6 TB/s).
constexpr int SQ_MOVERS = RT - 64;
template <class Tout> constexpr int SQ_E = 8192 / (int)sizeof(Tout);   // elements of a chunk, at most
template <class Tout> constexpr int SQ_K = SQ_E<Tout> / 64;            // one row: neighbours per lane
// a row of a chunk in LDS: 16 bytes after each row (or each lane's K
// elements) spread what the lanes read at once over the banks
template <class T, class Tout> constexpr int sq_pitch(int C, bool one) {
  return C + 16 / (int)sizeof(T) * (one ? C / SQ_K<Tout> : 1);
}

// lane l's v, in every lane
template <class T> __device__ inline T lane_value(T v, int l) {
  static_assert(sizeof(T) == 4 || sizeof(T) == 8, "one or two registers");
  int w[sizeof(T) / 4];
  __builtin_memcpy(w, &v, sizeof(T));
#pragma unroll
  for (int i = 0; i < (int)sizeof(T) / 4; i++) w[i] = __builtin_amdgcn_readlane(w[i], l);
  __builtin_memcpy(&v, w, sizeof(T));
  return v;
}

template <int OP, class Tin, class Tout, bool BAD, bool ONE>
__global__ __launch_bounds__(RT) void scan_seq(const Tin *__restrict__ a, RedPlan p, Outs o, BadInfo ba, int G, int C,
                                               int in_nfast, int out_nfast) {
  constexpr bool PR = (OP == R_CUMUPROD || OP == R_DCUMUPROD);
  constexpr int IT = 16, VI = 16 / (int)sizeof(Tin), VO = 16 / (int)sizeof(Tout);
  extern __shared__ __align__(16) char sq_lds[];
  const int pi = sq_pitch<Tin, Tout>(C, ONE), po = sq_pitch<Tout, Tout>(C, ONE);
  constexpr int K = SQ_K<Tout>;
  // [row offsets in a and in b][2 chunks of Tout][2 chunks of Tin]; pointers are
  // formed from sq_lds where they are used, which keeps them LDS pointers
  // (through a table of buffers they turn generic, and the scan three times slower)
  int64_t *rowa = (int64_t *)sq_lds, *rowb = rowa + G;
  auto out = [&](int64_t k) { return (Tout *)(sq_lds + 16 * G) + (int)(k & 1) * G * po; };
  auto in = [&](int64_t k) { return (Tin *)(sq_lds + 16 * G + 2 * G * po * sizeof(Tout)) + (int)(k & 1) * G * pi; };
  const int tid = threadIdx.x, lc = __builtin_ctz(C), lg = __builtin_ctz(G);
  const int64_t e0 = (int64_t)blockIdx.x * G;
  const int rows = p.nout - e0 < G ? (int)(p.nout - e0) : G;
  if (tid < rows) {
    int64_t off[MAXP];
    out_offsets(p, e0 + tid, off);
    rowa[tid] = off[0];
    rowb[tid] = off[1];
  }
  __syncthreads();
  const int64_t ia = p.inc_n[0], ib = p.inc_n[1], nc = (p.n + C - 1) / C;
  const Tin abv = bv_as<Tin>(ba.bv);
  const Tout obv = bv_as<Tout>(o.bv[0]);
  // position idx of a chunk -> row and element
  auto where = [&](int idx, int nfast, int &r, int &c) {
    r = nfast ? idx >> lc : idx & (G - 1);
    c = nfast ? idx & (C - 1) : idx >> lg;
  };
  // a mover's share of a chunk, all of its loads in flight at once (past the
  // rows' end the last element again: scanned after it, never stored)
  constexpr int U = SQ_E<Tout> / SQ_MOVERS + 1;
  const int me = tid - 64;
  Tin x[U];
  auto load = [&](int64_t k) {
    const int64_t c0 = k * C;
    const int clast = p.n - c0 < C ? (int)(p.n - c0) - 1 : C - 1;
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i = me + u * SQ_MOVERS;
      int r, c;
      where(i < G * C ? i : G * C - 1, in_nfast, r, c);
      x[u] = a[rowa[r < rows ? r : rows - 1] + (c0 + (c < clast ? c : clast)) * ia];
    }
  };
  auto commit = [&](int64_t k) {
    Tin *dst = in(k);
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i = me + u * SQ_MOVERS;
      int r, c;
      where(i, in_nfast, r, c);
      if (i < G * C) dst[ONE ? c + c / K * VI : r * pi + c] = x[u];
    }
  };
  auto store = [&](int64_t k) {
    const int64_t c0 = k * C;
    const int len = p.n - c0 < C ? (int)(p.n - c0) : C;
    const Tout *src = out(k);
    const auto bp = as_global((Tout *)o.p[0]);
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i = me + u * SQ_MOVERS;
      int r, c;
      where(i, out_nfast, r, c);
      if (i < G * C && r < rows && c < len) bp[rowb[r] + (c0 + c) * ib] = src[ONE ? c + c / K * VO : r * po + c];
    }
  };
  if (tid >= 64) {
    load(0);
    commit(0);
    if (nc > 1) load(1);
  }
  __syncthreads();
  Tout run = PR ? Tout(1) : Tout(0);
  for (int64_t k = 0; k <= nc; k++) {
    if (tid >= 64) {
      if (k + 1 < nc) commit(k + 1);
      if (k + 2 < nc) load(k + 2);
      if (k > 0) store(k - 1);
    } else if (ONE) {
      if (k < nc) {
        // what lies past the row's end is scanned last and not stored
        const int len = p.n - k * C < C ? (int)(p.n - k * C) : C;
        const Tin *src = in(k) + tid * (K + VI);
        Tout *dst = out(k) + tid * (K + VO);
        Tout v[K];
        unsigned skip = 0;
        if (tid * K < C) {
#pragma unroll
          for (int q = 0; q < K; q += VI) {
            const Vec<Tin, VI> t = *reinterpret_cast<const Vec<Tin, VI> *>(src + q);
#pragma unroll
            for (int i = 0; i < VI; i++) {
              v[q + i] = (Tout)t.v[i];
              if constexpr (BAD) skip |= isbad(t.v[i], abv, ba.isnan) ? 1u << (q + i) : 0u;
            }
          }
        }
        for (int l = 0; l * K < len; l++) {
          if (tid == l) {
#pragma unroll
            for (int i = 0; i < K; i++) {
              const Tout next = PR ? wmul(run, v[i]) : wadd(run, v[i]);
              const bool sk = BAD && (skip >> i & 1);
              run = sk ? run : next;
              v[i] = sk ? obv : run;
            }
          }
          run = lane_value(run, l);
        }
        if (tid * K < C) {
#pragma unroll
          for (int q = 0; q < K; q += VO) {
            Vec<Tout, VO> t;
#pragma unroll
            for (int i = 0; i < VO; i++) t.v[i] = v[q + i];
            *reinterpret_cast<Vec<Tout, VO> *>(dst + q) = t;
          }
        }
      }
    } else if (tid < rows && k < nc) {
      // whole groups of 16: what lies past the row's end is scanned last and not stored
      const Tin *src = in(k) + tid * pi;
      Tout *dst = out(k) + tid * po;
      const int len = p.n - k * C < C ? (int)(p.n - k * C) : C;
      Vec<Tin, VI> x[IT / VI];
#pragma unroll
      for (int v = 0; v < IT / VI; v++) x[v] = *reinterpret_cast<const Vec<Tin, VI> *>(src + v * VI);
      for (int c = 0; c < len; c += IT) {
        // 16 bytes of the wider type at a time: scan, store, and fetch the
        // elements of the next group that come to the same place.  In this
        // order an LDS access issues while the chain waits for its last sum.
        const int cn = c + IT < len ? c + IT : c;
        constexpr int VG = VI > VO ? VI : VO;
#pragma unroll
        for (int q = 0; q < IT; q += VG) {
          Vec<Tout, VO> y[VG / VO];
#pragma unroll
          for (int i = 0; i < VG; i++) {
            const Tin xi = x[(q + i) / VI].v[(q + i) % VI];
            bool skip = false;
            if constexpr (BAD) skip = isbad(xi, abv, ba.isnan);
            const Tout next = PR ? wmul(run, (Tout)xi) : wadd(run, (Tout)xi);
            run = skip ? run : next;
            y[i / VO].v[i % VO] = skip ? obv : run;
          }
#pragma unroll
          for (int v = 0; v < VG / VO; v++) *reinterpret_cast<Vec<Tout, VO> *>(dst + c + q + v * VO) = y[v];
#pragma unroll
          for (int v = 0; v < VG / VI; v++)
            x[q / VI + v] = *reinterpret_cast<const Vec<Tin, VI> *>(src + cn + q + v * VI);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    __syncthreads();
  }
}

template <int OP, class Tin, class Tout, bool BAD>
static hipError_t seq_launch(const RedPlan &p, const Tin *a, const Outs &o, const BadInfo &ba, hipStream_t s) {
  // rows per block: two blocks per CU before a block takes a second row; 8 KiB
  // of outputs per chunk (37 KiB of LDS, four blocks per CU), no more than a
  // row has
  int G = 1;
  while (G < 64 && (int64_t)G * 2 * 512 <= p.nout) G *= 2;
  constexpr int E = SQ_E<Tout>;
  int C = E / G;
  while (C > 32 && C / 2 >= p.n) C /= 2;
  // more rows where they are short
  while (G < 64 && G * C * 2 <= E && (int64_t)G * 2 * 256 <= p.nout) G *= 2;
  // (the shortest rows: no more than a group of 16; 100000 of 16 ints 13.3 us,
  // 14.4 with 32)
  if (G > 1 && p.n <= 16) C = 16;
  const bool one = G == 1;
  auto mag = [](int64_t x) { return x < 0 ? -x : x; };
  auto nfast = [&](int q) { return p.nout == 1 || p.nd == 0 || mag(p.inc_n[q]) <= mag(p.inc[q][0]); };
  const size_t lds = 16 * (size_t)G + 2 * (size_t)G * (sizeof(Tin) * sq_pitch<Tin, Tout>(C, one) +
                                                       sizeof(Tout) * sq_pitch<Tout, Tout>(C, one));
  const int64_t blocks = (p.nout + G - 1) / G;
  if (blocks >= GRID_BLOCKS) {   // two halves of the longest broadcast dim
    int d = 0;
    for (int k = 1; k < p.nd; k++) d = p.dims[k] > p.dims[d] ? k : d;
    RedPlan lo = p, hi = p;
    lo.dims[d] = p.dims[d] / 2;
    hi.dims[d] = p.dims[d] - lo.dims[d];
    lo.nout = p.nout / p.dims[d] * lo.dims[d];
    hi.nout = p.nout - lo.nout;
    for (int q = 0; q < p.npdl; q++) hi.off[q] += lo.dims[d] * p.inc[q][d];
    const hipError_t e = seq_launch<OP, Tin, Tout, BAD>(lo, a, o, ba, s);
    return e == hipSuccess ? seq_launch<OP, Tin, Tout, BAD>(hi, a, o, ba, s) : e;
  }
  const dim3 grid((unsigned)blocks);
  if (one)
    hipLaunchKernelGGL((scan_seq<OP, Tin, Tout, BAD, true>), grid, dim3(RT), lds, s, a, p, o, ba, G, C,
                       nfast(0) ? 1 : 0, nfast(1) ? 1 : 0);
  else
    hipLaunchKernelGGL((scan_seq<OP, Tin, Tout, BAD, false>), grid, dim3(RT), lds, s, a, p, o, ba, G, C,
                       nfast(0) ? 1 : 0, nfast(1) ? 1 : 0);
  return hipGetLastError();
}

// ---------------------------------------------------------------- thread
template <int OP, class Tin, class Tout, class Tacc, bool BAD>
__global__ __launch_bounds__(RT) void red_thread(const Tin *__restrict__ a, RedPlan p, Outs o, BadInfo ba,
                                                 int *flag) {
  const Tin abv = bv_as<Tin>(ba.bv);
  for (int64_t e = (int64_t)blockIdx.x * RT + threadIdx.x; e < p.nout; e += (int64_t)gridDim.x * RT) {
    int64_t off[MAXP];
    out_offsets(p, e, off);
    const Tin *ap = a + off[0];
    const int64_t n = p.n, ia = p.inc_n[0];
    if constexpr (OP == R_MIN_N_IND || OP == R_MAX_N_IND) {
      // Ufunc.pd:484-540: m passes, each skipping indices already chosen
      int64_t *cp = (int64_t *)o.p[0] + off[1];
      const int64_t ic = p.inc_m, m = p.m;
      const int64_t cbv = bv_as<int64_t>(o.bv[0]);
      Tin cur = 0;
      for (int64_t mi = 0; mi < m; mi++) {
        int64_t curind = n;
        for (int64_t i = 0; i < n; i++) {
          bool taken = false;
          for (int64_t mm = 0; mm < mi; mm++) if (cp[mm * ic] == i) { taken = true; break; }
          if (taken) continue;
          Tin x = ap[i * ia];
          if (BAD && isbad(x, abv, ba.isnan)) continue;
          bool better = (OP == R_MIN_N_IND) ? (x < cur) : (x > cur);
          if (curind == n || better || is_nan(cur)) { cur = x; curind = i; }
        }
        if (curind != n) cp[mi * ic] = curind;
        else {
          cp[mi * ic] = cbv;
          // PDL clears c's bad flag at the start of every broadcast iteration
          // and sets it on a shortfall, so the last iteration decides
          if (flag && e == p.nout - 1) atomicOr(flag, 1);
        }
      }
    } else if constexpr (is_prod(OP) && IsFloat<Tacc>::v) {
      // Ufunc.pd:104-108: sequential, stop at a zero running product
      Tacc tmp = 1;
      bool any = false;
      for (int64_t i = 0; i < n; i++) {
        Tin x = ap[i * ia];
        if constexpr (BAD) { if (isbad(x, abv, ba.isnan)) continue; }
        any = true;
        tmp *= (Tacc)x;
        if (tmp == 0) break;
      }
      Tout v = (Tout)tmp;
      if (BAD && !any) v = bv_as<Tout>(o.bv[0]);
      put<Tout>(o.p[0], off[1], v);
    } else {
      Part<Tin, Tacc> pt;
      part_init<OP, Tin, Tacc>(pt);
      for (int64_t i = 0; i < n; i++) {
        const Tin x = ap[i * ia];
        if constexpr (BAD) { if (isbad(x, abv, ba.isnan)) continue; }
        part_push<OP, Tin, Tacc>(pt, x, i);
      }
      part_store<OP, Tin, Tout, Tacc>(pt, o, off, BAD);
    }
  }
}

template <int OP, class Tin, class Tout, class Tacc, bool BAD>
static hipError_t thread_launch(const RedPlan &p, const Tin *a, const Outs &o, const BadInfo &ba, int *flag,
                                hipStream_t s) {
  int64_t blocks = (p.nout + RT - 1) / RT;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL((red_thread<OP, Tin, Tout, Tacc, BAD>), dim3((unsigned)blocks), dim3(RT), 0, s, a, p, o, ba, flag);
  return hipGetLastError();
}

// ---------------------------------------------------------------- dispatch
// launches red_grid: lanes along n where its stride is the smaller of the
// two, a wave's worth of outputs side by side otherwise; n is cut into chunks
// of at least 32 elements per thread until there are about 1024 blocks (four
// per CU; 2048 measured 22.5 + 7.0 us for that table).  Where memory for the
// partials cannot be had, n stays whole and the call still runs.
template <int OP, class Tin, class Tout, class Tacc, bool BAD>
static hipError_t grid_launch(const RedPlan &p, const Tin *a, const Outs &o, const BadInfo &ba, hipStream_t s) {
  const int64_t in0 = p.inc_n[0] < 0 ? -p.inc_n[0] : p.inc_n[0];
  const int64_t ie0 = p.nd == 0 || p.nout == 1 ? INT64_MAX : (p.inc[0][0] < 0 ? -p.inc[0][0] : p.inc[0][0]);
  const bool nfast = in0 < ie0;
  // The shortest rows, and short columns of outputs that fill the chip: the
  // plain loop of red_thread, whose block holds nothing but its outputs
  // (1000000 rows of 5 floats 8 us, here 12; 3000000 columns of 10 floats 29,
  // here 35; rows of 8 doubles 24 and 17, columns of 33 doubles 20 and 17).
  if (nfast ? p.n < 8 || p.n * (int64_t)sizeof(Tin) <= 16 : p.n < 16 && p.nout >= 262144)
    return thread_launch<OP, Tin, Tout, Tacc, BAD>(p, a, o, ba, nullptr, s);
  int LE, R;
  if (nfast) {
    // a thread for rows up to 64 bytes, then one for every 16 elements: with
    // fewer to load, the tree costs a thread more than it saves (1000000 rows
    // of 63 floats: 63 us, with a thread per four elements 187; of 16 floats
    // 33 and 44)
    R = 1;
    if (p.n * (int64_t)sizeof(Tin) > 64)
      while (R < 64 && R * 16 <= p.n) R *= 2;
    LE = RT / R;
    if (p.nout < LE) {   // fewer outputs than that: more threads along n
      LE = (int)p.nout;
      while (R * 2 * LE <= RT && R * 4 < p.n) R *= 2;
    }
  } else {
    // a thread per output where n is short or the outputs alone fill the chip
    // (256896 columns of 11 doubles: 7 us, 500000 of 100 floats: 33; with four
    // threads each 11 and 38 to 45)
    LE = p.nout < 64 ? (int)p.nout : p.n <= 32 || p.nout >= 262144 ? RT : 64;
    R = RT / LE;
  }
  const int64_t ngroup = (p.nout + LE - 1) / LE;
  int64_t nchunk = (1024 + ngroup - 1) / ngroup;
  const int64_t most = p.n / ((int64_t)R * 32);
  nchunk = nchunk < most ? nchunk : most;
  static_assert(sizeof(Part<Tin, Tacc>) <= 56, "the caller's scratch counts on it");
  Part<Tin, Tacc> *parts = nullptr;
  if (nchunk > 1) {
    const size_t need = sizeof(*parts) * (size_t)p.nout * (size_t)nchunk;
    if (p.scratch && need > (size_t)p.scratch_bytes) return hipErrorOutOfMemory;
    parts = (Part<Tin, Tacc> *)(p.scratch ? p.scratch : partials_alloc(need));
    if (!parts) nchunk = 1;
  } else {
    nchunk = 1;
  }
  int64_t clen = (p.n + nchunk - 1) / nchunk;
  clen = clen < 1 ? 1 : clen;
  const int64_t blocks = (ngroup < (1 << 20) ? ngroup : (1 << 20)) * nchunk;
  if (nfast)
    hipLaunchKernelGGL((red_grid<OP, Tin, Tout, Tacc, BAD, true>), dim3((unsigned)blocks), dim3(RT), 0, s, a, p, o, ba,
                       LE, R, nchunk, clen, parts);
  else
    hipLaunchKernelGGL((red_grid<OP, Tin, Tout, Tacc, BAD, false>), dim3((unsigned)blocks), dim3(RT), 0, s, a, p, o,
                       ba, LE, R, nchunk, clen, parts);
  if (parts) split2_launch<OP, Tin, Tout, Tacc, BAD>(p, nchunk, parts, o, s);
  const hipError_t err = hipGetLastError();
  if (parts && !p.scratch) partials_free(parts);
  return err;
}

template <int OP, class Tin, class Tout, class Tacc, bool BAD>
static hipError_t red_launch(const RedPlan &p, const Tin *a, const Outs &o, const BadInfo &ba, int *flag,
                             hipStream_t s) {
  if (p.nout == 0) return hipSuccess;
  constexpr bool SCAN = (OP == R_CUMUSUM || OP == R_DCUMUSUM || OP == R_CUMUPROD || OP == R_DCUMUPROD);
  constexpr bool SEQ = SCAN || OP == R_MIN_N_IND || OP == R_MAX_N_IND || (is_prod(OP) && IsFloat<Tacc>::v);
  if constexpr (!SEQ) {
    if (p.n >= 64 && p.inc_n[0] == 1) {
      const bool stream = streaming_read((size_t)p.n * (size_t)p.nout * sizeof(Tin));
      const size_t row_bytes = (size_t)p.n * sizeof(Tin);
      if (p.nout < 512 && row_bytes >= ((size_t)512 << 10)) {
        // long rows, few outputs: about 2048 chunks in all, of 32 KiB or more
        int64_t want = (2048 + p.nout - 1) / p.nout;
        int64_t clen = (p.n + want - 1) / want;
        const int64_t least = (32 << 10) / (int64_t)sizeof(Tin);
        if (clen < least) clen = least;
        clen = (clen + RT - 1) / RT * RT;   // a multiple of the 16-byte vectors' length
        int64_t nchunk = (p.n + clen - 1) / clen;
        // partials in the caller's scratch when it brings one, else from the cache
        const size_t need = sizeof(Part<Tin, Tacc>) * (size_t)p.nout * (size_t)nchunk;
        Part<Tin, Tacc> *parts;
        if (p.scratch) {
          if (need > (size_t)p.scratch_bytes) return hipErrorOutOfMemory;
          parts = (Part<Tin, Tacc> *)p.scratch;
        } else {
          parts = (Part<Tin, Tacc> *)scratch_alloc(need);
          if (!parts) return hipErrorOutOfMemory;
        }
        hipLaunchKernelGGL((red_split1<OP, Tin, Tout, Tacc, BAD>), dim3((unsigned)(p.nout * nchunk)), dim3(RT), 0, s, a,
                           p, nchunk, clen, parts, ba, stream);
        split2_launch<OP, Tin, Tout, Tacc, BAD>(p, nchunk, parts, o, s);
        hipError_t err = hipGetLastError();
        if (!p.scratch) scratch_free(parts);
        return err;
      }
      // Waves per row: with more than about 5000 in all they run in turns and
      // only add their joining, so sixteen a row up to 256 rows, four up to
      // 1280, one beyond; more where a lane would have very many elements,
      // fewer where not even that many loads.  Both sides, us with 1 / 4 / 16:
      // maximum of 256 rows of 25600 shorts 23 / 10.6 / 7.7, 600 of 12800 floats
      // 15 / 9 / 20, 1500 of 8192 shorts 12.9 / 9.6, of 4096 floats 8.6 / 9.6,
      // 2676 of 2048 floats 7 / 13.5, 3500 of 1024 doubles 7 / 15.6, 2048 of
      // 51200 shorts 53 / 42 / 60.
      const int64_t loads = (int64_t)(row_bytes / 16 / 64), each = p.n / 64;   // per lane of one wave
      const int waves = (p.nout <= 256 && loads >= 32) || (p.nout <= 640 && each >= 1600) ? 16
                        : (p.nout <= 1280 && loads >= 8) || (p.nout <= 1600 && each >= 100) ||
                              (p.nout < 4096 && each >= 300)
                            ? 4
                            : 1;
      if (waves == 1) {
        int64_t blocks = (p.nout + 3) / 4;
        if (blocks > 65536) blocks = 65536;
        bool on16 = (uintptr_t)(a + p.off[0]) % 16 == 0;
        for (int d = 0; d < p.nd; d++) on16 = on16 && p.inc[0][d] * (int64_t)sizeof(Tin) % 16 == 0;
        if (on16)
          hipLaunchKernelGGL((red_wave<OP, Tin, Tout, Tacc, BAD, 1, true>), dim3((unsigned)blocks), dim3(RT), 0, s, a, p,
                             o, ba, stream);
        else
          hipLaunchKernelGGL((red_wave<OP, Tin, Tout, Tacc, BAD, 1>), dim3((unsigned)blocks), dim3(RT), 0, s, a, p, o,
                             ba, stream);
      } else if (waves == 4) {
        hipLaunchKernelGGL((red_wave<OP, Tin, Tout, Tacc, BAD, 4>), dim3((unsigned)p.nout), dim3(RT), 0, s, a, p, o, ba,
                           stream);
      } else {
        hipLaunchKernelGGL((red_wave<OP, Tin, Tout, Tacc, BAD, 16>), dim3((unsigned)p.nout), dim3(16 * 64), 0, s, a, p,
                           o, ba, stream);
      }
      return hipGetLastError();
    }
    return grid_launch<OP, Tin, Tout, Tacc, BAD>(p, a, o, ba, s);
  } else if constexpr (SCAN) {
    if constexpr ((OP == R_CUMUSUM || OP == R_CUMUPROD) && !IsFloat<Tout>::v) {
      if (p.inc_n[0] == 1 && p.inc_n[1] == 1 && p.n >= 256) {
        // rows of several chunks are cut while they alone leave CUs idle:
        // about 2048 blocks in all, each of at least 8192 elements.  From a
        // row per CU on, reading everything twice costs more (500 rows of
        // 40000 ints: 32 us, cut 43)
        int64_t nchunk = 1, clen = p.n;
        Tout *totals = nullptr;
        if (p.nout < 256 && p.n >= 32768) {
          int64_t want = (2048 + p.nout - 1) / p.nout;
          clen = (p.n + want - 1) / want;
          clen = clen < 8192 ? 8192 : (clen + SC_CH - 1) / SC_CH * SC_CH;
          nchunk = (p.n + clen - 1) / clen;
          totals = (Tout *)partials_alloc(sizeof(Tout) * (size_t)(p.nout * nchunk));
          if (!totals) { nchunk = 1; clen = p.n; }   // out of memory: a block per row
        }
        if (totals)
          hipLaunchKernelGGL((scan_totals<OP, Tin, Tout, BAD>), dim3((unsigned)(p.nout * nchunk)), dim3(RT), 0, s, a, p,
                             ba, nchunk, clen, totals);
        const int64_t blocks = p.nout * nchunk < 65536 ? p.nout * nchunk : 65536;
        if (totals)
          hipLaunchKernelGGL((scan_rows<OP, Tin, Tout, BAD, true>), dim3((unsigned)blocks), dim3(RT), 0, s, a, p, o, ba,
                             nchunk, clen, totals);
        else
          hipLaunchKernelGGL((scan_rows<OP, Tin, Tout, BAD, false>), dim3((unsigned)blocks), dim3(RT), 0, s, a, p, o, ba,
                             nchunk, clen, totals);
        const hipError_t err = hipGetLastError();
        if (totals) partials_free(totals);
        return err;
      }
    }
    if (p.n == 0) return hipSuccess;
    return seq_launch<OP, Tin, Tout, BAD>(p, a, o, ba, s);
  } else {
    return thread_launch<OP, Tin, Tout, Tacc, BAD>(p, a, o, ba, flag, s);
  }
}

template <int OP, class Tin, class Tout, class Tacc>
static hipError_t red_bad(bool bad, const RedPlan &p, const Tin *a, const Outs &o, const BadInfo &ba, int *flag,
                          hipStream_t s) {
  return bad ? red_launch<OP, Tin, Tout, Tacc, true>(p, a, o, ba, flag, s)
             : red_launch<OP, Tin, Tout, Tacc, false>(p, a, o, ba, flag, s);
}

template <class Tin>
static hipError_t reduce_T(int op, const RedPlan &p, const void *va, void *const *outs, bool bad, const BadInfo &ba,
                           const pdlhip_value *obv, int *flag, hipStream_t s) {
  typedef typename IPlus<Tin>::O TI;
  const Tin *a = (const Tin *)va;
  Outs o;
  for (int k = 0; k < 4; k++) { o.p[k] = outs[k]; o.bv[k] = obv[k]; }
  switch (op) {
  case R_SUM: return red_bad<R_SUM, Tin, TI, TI>(bad, p, a, o, ba, flag, s);
  case R_PROD: return red_bad<R_PROD, Tin, TI, TI>(bad, p, a, o, ba, flag, s);
  case R_DSUM: return red_bad<R_DSUM, Tin, double, double>(bad, p, a, o, ba, flag, s);
  case R_DPROD: return red_bad<R_DPROD, Tin, double, double>(bad, p, a, o, ba, flag, s);
  case R_CUMUSUM: return red_bad<R_CUMUSUM, Tin, TI, TI>(bad, p, a, o, ba, flag, s);
  case R_CUMUPROD: return red_bad<R_CUMUPROD, Tin, TI, TI>(bad, p, a, o, ba, flag, s);
  case R_DCUMUSUM: return red_bad<R_DCUMUSUM, Tin, double, double>(bad, p, a, o, ba, flag, s);
  case R_DCUMUPROD: return red_bad<R_DCUMUPROD, Tin, double, double>(bad, p, a, o, ba, flag, s);
  case R_AVERAGE: return red_bad<R_AVERAGE, Tin, TI, TI>(bad, p, a, o, ba, flag, s);
  case R_DAVERAGE: return red_bad<R_DAVERAGE, Tin, double, double>(bad, p, a, o, ba, flag, s);
  case R_MIN: return red_bad<R_MIN, Tin, Tin, Tin>(bad, p, a, o, ba, flag, s);
  case R_MAX: return red_bad<R_MAX, Tin, Tin, Tin>(bad, p, a, o, ba, flag, s);
  case R_MIN_IND: return red_bad<R_MIN_IND, Tin, int64_t, Tin>(bad, p, a, o, ba, flag, s);
  case R_MAX_IND: return red_bad<R_MAX_IND, Tin, int64_t, Tin>(bad, p, a, o, ba, flag, s);
  case R_MINMAXIMUM: return red_bad<R_MINMAXIMUM, Tin, Tin, Tin>(bad, p, a, o, ba, flag, s);
  case R_MIN_N_IND: return red_bad<R_MIN_N_IND, Tin, int64_t, Tin>(bad, p, a, o, ba, flag, s);
  case R_MAX_N_IND: return red_bad<R_MAX_N_IND, Tin, int64_t, Tin>(bad, p, a, o, ba, flag, s);
  default: return hipErrorInvalidValue;
  }
}

#define PDLHIP_RED_TYPE(TC) \
  hipError_t launch_reduce_t##TC(int op, int otype, const RedPlan &p, const void *a, void *const *outs, bool bad, \
                                 const BadInfo &ba, const pdlhip_value *obv, int *flag, hipStream_t s) { \
    (void)otype; \
    return reduce_T<CType<TC>::T>(op, p, a, outs, bad, ba, obv, flag, s); \
  }
PDLHIP_RED_TYPES_IN_THIS_TU

}  // namespace pdlhip
