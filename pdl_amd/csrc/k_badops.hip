// Bad.pd's elementwise ops over a canonical plan (the reference's loops:
// lib/PDL/Bad.pd:343-395 isbad/isgood, 584-634 setbadif, 639-676
// setvaltobad, 679-775 setnantobad/setinftobad/setnonfinitetobad, 777-806
// setbadtonan, 808-840 setbadtoval).
//
// $ISBAD(x) compiles to PDL_ISBAD2(x, x_badval, ...) in the good and the bad
// code alike (PP/PDLCode.pm:664-668); only PDL_IF_BAD(t, f) depends on the
// trans's bvalflag.  So setbadtonan and setvaltobad test values in both
// modes, isbad/isgood/setbadif/setbadtoval only in bad mode.
//
// Grid-stride loops; the plan orders dims by the output's strides, so
// consecutive threads write consecutive elements.  The ops that set the output's bad flag only when they found something
// (setnantobad, setinftobad, setnonfinitetobad) raise a device flag the host
// reads back.
#include <hip/hip_runtime.h>

#include "device.hpp"
#include "launch.hpp"

namespace pdlhip {

constexpr int BADOP_THREADS = 256;

template <class T> __device__ inline bool finite_v(T v) {
  if constexpr (IsFloat<T>::v) return isfinite(v);
  else return true;
}

// one element; hit where an op found a value to set bad
template <class T, class To, int OP>
__device__ __forceinline__ To bad_one(T x, int32_t mk, T abv, const BadInfo &ba, int32_t mbv, To bbv, T val, int bad,
                                      bool &hit) {
  if constexpr (OP == B_ISBAD) {
    return (To)(bad ? isbad(x, abv, ba.isnan) : 0);
  } else if constexpr (OP == B_ISGOOD) {
    return (To)(bad ? !isbad(x, abv, ba.isnan) : 1);
  } else if constexpr (OP == B_SETBADIF) {
    return ((bad && mk == mbv) || mk) ? bbv : (To)x;
  } else if constexpr (OP == B_SETVALTOBAD) {
    return (x == val) ? bbv : (To)x;
  } else if constexpr (OP == B_SETNANTOBAD || OP == B_SETINFTOBAD || OP == B_SETNONFINITETOBAD) {
    bool set;
    if constexpr (OP == B_SETNANTOBAD) set = is_nan(x);
    else if constexpr (OP == B_SETINFTOBAD) set = !finite_v(x) && !is_nan(x);
    else set = !finite_v(x);
    hit |= set;
    return set ? bbv : (To)x;
  } else if constexpr (OP == B_SETBADTONAN) {
    return isbad(x, abv, ba.isnan) ? (To)__builtin_nan("") : (To)x;
  } else {
    static_assert(OP == B_SETBADTOVAL, "a Bad.pd elementwise op");
    return (bad && isbad(x, abv, ba.isnan)) ? (To)val : (To)x;
  }
}

// any plan, an element per thread per step
template <class T, class To, int OP>
__global__ __launch_bounds__(BADOP_THREADS) void bad_ew(const T *__restrict__ a, const int32_t *__restrict__ m,
                                                        To *__restrict__ b, EwPlan p, BadInfo ba, int32_t mbv,
                                                        To bbv, T val, int bad, int *flag) {
  const T abv = bv_as<T>(ba.bv);
  bool hit = false;
  for (int64_t e = (int64_t)blockIdx.x * BADOP_THREADS + threadIdx.x; e < p.n;
       e += (int64_t)gridDim.x * BADOP_THREADS) {
    int64_t r = e, o0 = p.off[0], o1 = p.off[1], o2 = p.off[2];
    for (int d = 0; d < p.nd; d++) {
      // one dim, or the last: what is left of e is its index (no division)
      const int64_t i = d == p.nd - 1 ? r : r % p.dims[d];
      if (d < p.nd - 1) r /= p.dims[d];
      o0 += i * p.inc[0][d];
      o1 += i * p.inc[1][d];
      o2 += i * p.inc[2][d];
    }
    b[o2] = bad_one<T, To, OP>(a[o0], OP == B_SETBADIF ? m[o1] : 0, abv, ba, mbv, bbv, val, bad, hit);
  }
  if (hit) *flag = 1;   // the same value from every writer
}

// contiguous, 16-byte aligned operands (the mask contiguous or one element):
// V elements per load, two loads in flight per thread.  Bound by HBM: 8192^2
// shorts with the element-wise kernel took 126 us (isgood, 3.2 TB/s) and 106
// us (setbadtoval, 2.5 TB/s), most of it dividing 64-bit positions; this
// takes 72 us (5.6 TB/s) and 38 us (7.1 TB/s, much of it from the cache).
template <class T> struct BadVec { static constexpr int V = sizeof(T) == 1 ? 8 : 16 / (int)sizeof(T); };

template <class T, class To, int OP>
__global__ __launch_bounds__(BADOP_THREADS) void bad_flat(const T *__restrict__ a, const int32_t *__restrict__ m,
                                                          To *__restrict__ b, int64_t n, int minc, BadInfo ba,
                                                          int32_t mbv, To bbv, T val, int bad, int *flag) {
  constexpr int V = BadVec<T>::V, U = 2;
  constexpr int VS = V * (int)sizeof(To) <= 16 ? V : 16 / (int)sizeof(To);   // elements per store
  constexpr int VM = V < 4 ? V : 4;                                            // mask elements per load
  const T abv = bv_as<T>(ba.bv);
  const int32_t m0 = OP == B_SETBADIF && !minc ? m[0] : 0;
  bool hit = false;
  const int64_t nv = n / V, stride = (int64_t)gridDim.x * BADOP_THREADS;
  for (int64_t g = (int64_t)blockIdx.x * BADOP_THREADS + threadIdx.x; g < nv; g += U * stride) {
    Vec<T, V> x[U];
    int32_t mk[U][V];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int64_t q = g + u * stride < nv ? g + u * stride : g;
      x[u] = *reinterpret_cast<const Vec<T, V> *>(a + q * V);
      if constexpr (OP == B_SETBADIF) {
#pragma unroll
        for (int k = 0; k < V; k += VM) {
          Vec<int32_t, VM> mv;
          if (minc) mv = *reinterpret_cast<const Vec<int32_t, VM> *>(m + q * V + k);
#pragma unroll
          for (int i = 0; i < VM; i++) mk[u][k + i] = minc ? mv.v[i] : m0;
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (g + u * stride >= nv) break;
#pragma unroll
      for (int k = 0; k < V; k += VS) {
        Vec<To, VS> y;
#pragma unroll
        for (int i = 0; i < VS; i++)
          y.v[i] = bad_one<T, To, OP>(x[u].v[k + i], OP == B_SETBADIF ? mk[u][k + i] : 0, abv, ba, mbv, bbv, val, bad, hit);
        *reinterpret_cast<Vec<To, VS> *>(b + (g + u * stride) * V + k) = y;
      }
    }
  }
  const int64_t t = nv * V + threadIdx.x;   // the rest, fewer than V
  if (blockIdx.x == 0 && t < n)
    b[t] = bad_one<T, To, OP>(a[t], OP == B_SETBADIF ? (minc ? m[t] : m0) : 0, abv, ba, mbv, bbv, val, bad, hit);
  if (hit) *flag = 1;
}

template <class T, class To, int OP>
static hipError_t bad_go(const EwPlan &p, const void *a, const void *m, void *b, const BadInfo &ba, int32_t mbv,
                         const pdlhip_value &bbv, double dval, bool bad, int *flag, hipStream_t s) {
  // $GENERIC(a) $COMP(value): the double OtherPar in the trans type, as C converts it
  const T val = (T)dval;
  const T *pa = (const T *)a + p.off[0];
  const int32_t *pm = OP == B_SETBADIF ? (const int32_t *)m + p.off[1] : nullptr;
  To *pb = (To *)b + p.off[2];
  auto on16 = [](const void *q) { return (uintptr_t)q % 16 == 0; };
  if (p.nd == 1 && p.inc[0][0] == 1 && p.inc[2][0] == 1 && on16(pa) && on16(pb) &&
      (OP != B_SETBADIF || p.inc[1][0] == 0 || (p.inc[1][0] == 1 && on16(pm)))) {
    const int64_t per = (int64_t)BADOP_THREADS * BadVec<T>::V * 2;
    int64_t grid = (p.n + per - 1) / per;
    grid = grid < 1 ? 1 : (grid > 65536 ? 65536 : grid);
    hipLaunchKernelGGL((bad_flat<T, To, OP>), dim3((unsigned)grid), dim3(BADOP_THREADS), 0, s, pa, pm, pb, p.n,
                       (int)p.inc[1][0], ba, mbv, bv_as<To>(bbv), val, bad ? 1 : 0, flag);
    return hipGetLastError();
  }
  int64_t grid = (p.n + BADOP_THREADS * 4 - 1) / (BADOP_THREADS * 4);
  grid = grid < 1 ? 1 : (grid > 65536 ? 65536 : grid);
  hipLaunchKernelGGL((bad_ew<T, To, OP>), dim3((unsigned)grid), dim3(BADOP_THREADS), 0, s, (const T *)a,
                     (const int32_t *)m, (To *)b, p, ba, mbv, bv_as<To>(bbv), val, bad ? 1 : 0, flag);
  return hipGetLastError();
}

template <class T>
static hipError_t bad_T(int op, const EwPlan &p, const void *a, const void *m, void *b, const BadInfo &ba,
                        int32_t mbv, const pdlhip_value &bbv, double dval, bool bad, int *flag, hipStream_t s) {
  switch (op) {
  case B_ISBAD: return bad_go<T, int32_t, B_ISBAD>(p, a, m, b, ba, mbv, bbv, dval, bad, flag, s);
  case B_ISGOOD: return bad_go<T, int32_t, B_ISGOOD>(p, a, m, b, ba, mbv, bbv, dval, bad, flag, s);
  case B_SETBADIF: return bad_go<T, T, B_SETBADIF>(p, a, m, b, ba, mbv, bbv, dval, bad, flag, s);
  case B_SETVALTOBAD: return bad_go<T, T, B_SETVALTOBAD>(p, a, m, b, ba, mbv, bbv, dval, bad, flag, s);
  case B_SETBADTOVAL: return bad_go<T, T, B_SETBADTOVAL>(p, a, m, b, ba, mbv, bbv, dval, bad, flag, s);
  default: break;
  }
  if constexpr (IsFloat<T>::v) {
    switch (op) {
    case B_SETNANTOBAD: return bad_go<T, T, B_SETNANTOBAD>(p, a, m, b, ba, mbv, bbv, dval, bad, flag, s);
    case B_SETINFTOBAD: return bad_go<T, T, B_SETINFTOBAD>(p, a, m, b, ba, mbv, bbv, dval, bad, flag, s);
    case B_SETNONFINITETOBAD:
      return bad_go<T, T, B_SETNONFINITETOBAD>(p, a, m, b, ba, mbv, bbv, dval, bad, flag, s);
    case B_SETBADTONAN: return bad_go<T, T, B_SETBADTONAN>(p, a, m, b, ba, mbv, bbv, dval, bad, flag, s);
    default: break;
    }
  }
  return hipErrorInvalidValue;
}

hipError_t launch_badop(int T, int op, const EwPlan &p, const void *a, const void *m, void *b, const BadInfo &ba,
                        int32_t mbv, const pdlhip_value &bbv, double dval, bool bad, int *flag, hipStream_t s) {
  switch (T) {
#define X(TC) case TC: return bad_T<CType<TC>::T>(op, p, a, m, b, ba, mbv, bbv, dval, bad, flag, s);
    PDLHIP_FOR_EACH_TYPE(X)
#undef X
  default: return hipErrorInvalidValue;
  }
}

}  // namespace pdlhip
