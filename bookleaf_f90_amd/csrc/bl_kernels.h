// bl_kernels.h -- deterministic workgroup reductions used by the dt controls.
//
// hydro_kn_getdtcfl picks the FIRST element attaining the minimum of
// rscratch11 (strict '<' scan, hydro_kn_getdt.f90:68-72); hydro_kn_getdtdiv
// picks the FIRST element attaining the maximum, and only if it exceeds TINY
// (strict '>' scan from TINY, hydro_kn_getdt.f90:104-117).  Both are total
// orders on (value, index), so a tree reduction in any order returns the
// same element as the serial scan: register moves across a wave, LDS across
// the waves of the workgroup, then one workgroup over the partials (a step on
// a small tiling: every tile).
#pragma once
#include <hip/hip_runtime.h>
#include <cfloat>

#include "bl_internal.h"

namespace bl {

__device__ __forceinline__ void better_min(double& v, int& i, double v2, int i2) {
  if (v2 < v || (v2 == v && i2 < i)) { v = v2; i = i2; }
}
__device__ __forceinline__ void better_max(double& v, int& i, double v2, int i2) {
  if (v2 > v || (v2 == v && i2 < i)) { v = v2; i = i2; }
}

// The wave's reductions move data between lanes with data-parallel
// primitives (a register move each) rather than shuffles (a trip through the
// LDS unit each, which a reduction waits for six times): row_shr 1, 2, 4 and 8
// within the rows of 16, then row_bcast 15 and 31 across them, which leaves
// the result in lane 63.  A lane that reads none keeps its own value.  The
// Sedov step's tile kernel, whose workgroups each end with two of them, went
// from 77 to 74 us, the 200x20 Sod step from 25.7 to 23.7 us.
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_move(int x) {
  return __builtin_amdgcn_update_dpp(x, x, CTRL, ROWS, 0xf, false);
}
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_move(double x) {
  const int2 h = __builtin_bit_cast(int2, x);
  return __builtin_bit_cast(double, make_int2(dpp_move<CTRL, ROWS>(h.x), dpp_move<CTRL, ROWS>(h.y)));
}
template <typename T, typename OP>
__device__ __forceinline__ T wave_fold(T x, OP op) {
  x = op(x, dpp_move<0x111, 0xf>(x));
  x = op(x, dpp_move<0x112, 0xf>(x));
  x = op(x, dpp_move<0x114, 0xf>(x));
  x = op(x, dpp_move<0x118, 0xf>(x));
  x = op(x, dpp_move<0x142, 0xa>(x));
  x = op(x, dpp_move<0x143, 0xc>(x));
  return x;
}
__device__ __forceinline__ int lane_value(int x, int lane) {
  return __builtin_amdgcn_readlane(x, lane);
}
__device__ __forceinline__ double lane_value(double x, int lane) {
  const int2 h = __builtin_bit_cast(int2, x);
  return __builtin_bit_cast(double, make_int2(lane_value(h.x, lane), lane_value(h.y, lane)));
}

// the wave's inclusive prefix sum (whole waves only)
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp_or_zero(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, ROWS, 0xf, false);
}
__device__ __forceinline__ uint32_t wave_prefix(uint32_t x) {
  x += dpp_or_zero<0x111, 0xf>(x);
  x += dpp_or_zero<0x112, 0xf>(x);
  x += dpp_or_zero<0x114, 0xf>(x);
  x += dpp_or_zero<0x118, 0xf>(x);
  x += dpp_or_zero<0x142, 0xa>(x);
  x += dpp_or_zero<0x143, 0xc>(x);
  return x;
}

// the wave's first-index minimum (maximum) of (v, i), in every lane: the
// extreme value, the smallest index that has it, and that lane's own value
// (whole waves only; no NaN)
template <bool IS_MIN>
__device__ __forceinline__ void wave_reduce(double& v, int& i) {
  const double m = lane_value(
      wave_fold(v, [](double a, double b) { return (IS_MIN ? b < a : b > a) ? b : a; }), 63);
  const int k = lane_value(wave_fold(v == m ? i : 0x7fffffff, [](int a, int b) { return b < a ? b : a; }), 63);
  const uint64_t who = __ballot(v == m && i == k);
  v = lane_value(v, __ffsll((unsigned long long)who) - 1);
  i = k;
}

// reduce over the workgroup; thread 0 writes the result to (*outv, *outi)
template <bool IS_MIN>
__device__ __forceinline__ void block_reduce_at(double v, int i, double* outv, int32_t* outi) {
  __shared__ double sv[kBlock / 64];
  __shared__ int si[kBlock / 64];
  wave_reduce<IS_MIN>(v, i);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) { sv[wid] = v; si[wid] = i; }
  __syncthreads();
  if (threadIdx.x == 0) {
    double bv = sv[0];
    int bi = si[0];
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) {
      if (IS_MIN) better_min(bv, bi, sv[w], si[w]);
      else better_max(bv, bi, sv[w], si[w]);
    }
    *outv = bv;
    *outi = bi;
  }
}

// the DIV maximum (dv, di) and the CFL minimum (cv, ci) over the workgroup
// together, one barrier for both; thread 0 writes them
__device__ __forceinline__ void block_reduce_div_cfl(double dv, int di, double cv, int ci,
                                                     double* out_dv, int32_t* out_di,
                                                     double* out_cv, int32_t* out_ci) {
  __shared__ double sv[2][kBlock / 64];
  __shared__ int si[2][kBlock / 64];
  wave_reduce<false>(dv, di);
  wave_reduce<true>(cv, ci);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) {
    sv[0][wid] = dv; si[0][wid] = di;
    sv[1][wid] = cv; si[1][wid] = ci;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) {
      better_max(dv, di, sv[0][w], si[0][w]);
      better_min(cv, ci, sv[1][w], si[1][w]);
    }
    *out_dv = dv; *out_di = di;
    *out_cv = cv; *out_ci = ci;
  }
}

// the partial of this workgroup at part[blockIdx.x]
template <bool IS_MIN>
__device__ __forceinline__ void block_reduce_store(double v, int i, double* part, int32_t* parti) {
  block_reduce_at<IS_MIN>(v, i, part + blockIdx.x, parti + blockIdx.x);
}

__device__ __forceinline__ void block_argmin_first(double v, int i, double* part, int32_t* parti) {
  if (!(v == v)) v = DBL_MAX;  // a NaN never wins the strict '<' scan
  block_reduce_store<true>(v, i, part, parti);
}
__device__ __forceinline__ void block_argmax_first(double v, int i, double* part, int32_t* parti) {
  if (!(v == v)) v = -1.0;  // a NaN never wins the strict '>' scan
  block_reduce_store<false>(v, i, part, parti);
}

// run by one workgroup of up to kFinalBlock threads: DIV partials in
// part[0,na), CFL partials in part[2na, 2na+nc); both in one pass so the
// loads of a thread are independent
constexpr int kFinalBlock = 1024;
// this thread's share of the DIV partials (part, parti)[0, na) and the CFL
// partials (pc, qc)[0, nc): DIV maximum (va, xa), CFL minimum (vc, xc)
__device__ __forceinline__ void final_dt_gather(int na, const double* part, const int32_t* parti,
                                                int nc, const double* pc, const int32_t* qc,
                                                double& va, int& xa, double& vc, int& xc) {
  va = -1.0; vc = DBL_MAX;
  xa = 0x7fffffff; xc = 0x7fffffff;
  const int nmax = na > nc ? na : nc;
  if (na < 1 || nc < 1) {  // (not a case the step launches)
    for (int k = threadIdx.x; k < nmax; k += blockDim.x) {
      if (k < na) better_max(va, xa, part[k], parti[k]);
      if (k < nc) better_min(vc, xc, pc[k], qc[k]);
    }
    return;
  }
  // kPer entries of each control per thread and pass, all loaded (from
  // clamped indices, so with no branch) before any is compared
  constexpr int kPer = 4;
  const int stride = (int)blockDim.x;
  for (int b = threadIdx.x; b < nmax; b += kPer * stride) {
    double a[kPer], c[kPer];
    int ai[kPer], ci[kPer];
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
      const int k = b + r * stride;
      const int ka = k < na ? k : na - 1, kc = k < nc ? k : nc - 1;
      a[r] = part[ka]; ai[r] = parti[ka];
      c[r] = pc[kc]; ci[r] = qc[kc];
    }
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
      const int k = b + r * stride;
      if (k < na) better_max(va, xa, a[r], ai[r]);
      if (k < nc) better_min(vc, xc, c[r], ci[r]);
    }
  }
}
// the workgroup's combination of the threads' shares into res
__device__ __forceinline__ void final_dt_combine(double va, int xa, double vc, int xc,
                                                 DtResult* res) {
  __shared__ double sa[kFinalBlock / 64], sc[kFinalBlock / 64];
  __shared__ int ia[kFinalBlock / 64], ic[kFinalBlock / 64];
  wave_reduce<false>(va, xa);
  wave_reduce<true>(vc, xc);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) { sa[wid] = va; ia[wid] = xa; sc[wid] = vc; ic[wid] = xc; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) {
      better_max(sa[0], ia[0], sa[w], ia[w]);
      better_min(sc[0], ic[0], sc[w], ic[w]);
    }
    if (sa[0] > DBL_MIN) { res->div_max = sa[0]; res->div_idx = ia[0]; }
    else { res->div_max = DBL_MIN; res->div_idx = 0; }
    res->cfl_min = sc[0];
    res->cfl_idx = ic[0];
  }
  __syncthreads();
}
// DIV partials (pa, qa)[0, na), CFL partials (pc, qc)[0, nc)
__device__ __forceinline__ void final_dt_reduce(int na, const double* part, const int32_t* parti,
                                                int nc, const double* pc, const int32_t* qc,
                                                DtResult* res) {
  double va, vc;
  int xa, xc;
  final_dt_gather(na, part, parti, nc, pc, qc, va, xa, vc, xc);
  final_dt_combine(va, xa, vc, xc, res);
}
__device__ __forceinline__ void final_dt_reduce(int na, int nc, const double* part,
                                                const int32_t* parti, DtResult* res) {
  final_dt_reduce(na, part, parti, nc, part + 2 * na, parti + 2 * na, res);
}

}  // namespace bl
