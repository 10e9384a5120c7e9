// bl_diag.hip -- conservation tables (hydro_dr_shortprint) and the Sod L1
// check (check_dr_tests / check_kn_sod) on the device.
//
// Reductions have a fixed shape: each workgroup reduces its elements per
// flag, across the lanes of each wave (wave_fold) and over its waves in LDS,
// then one workgroup per (flag, quantity) folds the workgroups' partials.
// Results are reproducible run to run and differ from the reference's serial
// sums only in rounding.
#include <hip/hip_runtime.h>

#include <cfloat>
#include <cstring>
#include <vector>

#include "bl_internal.h"
#include "bl_kernels.h"
#include "bl_math.h"
#include "bl_mix.h"

namespace bl {

// quantities of one table row, in bl_flag_totals_t order; 0-4 are sums,
// 5/7 minima, 6/8 maxima
constexpr int kNq = 9;

__device__ __forceinline__ double q_identity(int q) {
  return (q == 5 || q == 7) ? DBL_MAX : ((q == 6 || q == 8) ? -DBL_MAX : 0.0);
}
__device__ __forceinline__ double q_combine(int q, double a, double b) {
  if (q == 5 || q == 7) return dmin(a, b);
  if (q == 6 || q == 8) return dmax(a, b);
  return a + b;
}

// one element's contribution to its flag's row (hydro_kn_calc_shortprint,
// hydro_kn_print.F90:81-107); cu/cv the corner velocities
__device__ __forceinline__ void sp_row(double dencut, double den, double en, double pre,
                                       double vol, double mass, const double wt[4],
                                       const double cu[4], const double cv[4], double r[kNq]) {
  r[0] = vol;
  r[1] = 0.0; r[2] = 0.0; r[3] = 0.0; r[4] = 0.0;
  r[5] = DBL_MAX; r[6] = -DBL_MAX; r[7] = DBL_MAX; r[8] = -DBL_MAX;
  if (mass > dencut * vol) {
    r[1] = mass;
    r[2] = en * mass;
    r[4] = mass * pre;
    r[5] = pre; r[6] = pre; r[7] = den; r[8] = den;
    double ke = 0.0;
#pragma unroll
    for (int c = 0; c < 4; ++c) ke = 0.5 * wt[c] * den * (cu[c] * cu[c] + cv[c] * cv[c]) + ke;
    r[3] = ke;
  }
}

// the workgroup's combination of quantity q over its threads' v (thread 0 to
// kNq - 1 get one each, q = their own number): sh holds each wave's
__device__ __forceinline__ void wave_quantities(const double v[kNq], double sh[kNq]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int q = 0; q < kNq; ++q) {
    const double r = wave_fold(v[q], [q](double a, double b) { return q_combine(q, a, b); });
    if (lane == 63) sh[q] = r;
  }
}

// reduce r (this thread's contribution to flag `mine`, none if mine < 0)
// over the workgroup for every flag, into part[(f * kNq + q) * nb + b], b
// this workgroup's place among the nb.  Every thread of the workgroup must
// call it.
__device__ __forceinline__ void block_flag_reduce(int nflag, int mine, const double r[kNq],
                                                  int nb, int b, double* part) {
  __shared__ double sh[kBlock / 64][kNq];
  const int wid = threadIdx.x >> 6, t = threadIdx.x;
  for (int f = 0; f < nflag; ++f) {
    double v[kNq];
#pragma unroll
    for (int q = 0; q < kNq; ++q) v[q] = (mine == f) ? r[q] : q_identity(q);
    wave_quantities(v, sh[wid]);
    __syncthreads();
    if (t < kNq) {
      double x = sh[0][t];
      for (int w = 1; w < kBlock / 64; ++w) x = q_combine(t, x, sh[w][t]);
      part[((size_t)f * kNq + t) * nb + b] = x;
    }
    __syncthreads();
  }
}

// an element's row (hydro_kn_calc_shortprint) from its nodes' positions and
// velocities; its geometry in g
__device__ __forceinline__ void sp_row_nodes(double dencut, double den, double en, double pre,
                                             double mass, const double x[4], const double y[4],
                                             const double cu[4], const double cv[4], Iso& g,
                                             double r[kNq]) {
  getiso(x, y, g);
  sp_row(dencut, den, en, pre, g.vol, mass, g.wt, cu, cv, r);
}

// element rows by flag (ielreg or ielmat; flag <= 0 skipped), from the
// geometry fields; nb: the workgroups of the table (the components' come
// after the elements')
__global__ void __launch_bounds__(kBlock)
k_sp_elements(int nel, int nflag, double dencut, const int32_t* __restrict__ flag,
              const int32_t* __restrict__ ielnd, const double* __restrict__ den,
              const double* __restrict__ en, const double* __restrict__ pre,
              const double* __restrict__ vol, const double* __restrict__ mass,
              const double* __restrict__ cnwt, const double* __restrict__ ndu,
              const double* __restrict__ ndv, int nb, double* __restrict__ part) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  double r[kNq];
  int mine = -1;
  if (e < nel && flag[e] > 0) {
    mine = flag[e] - 1;
    const int4 q = reinterpret_cast<const int4*>(ielnd)[e];
    const int nd[4] = {q.x - 1, q.y - 1, q.z - 1, q.w - 1};
    const double cu[4] = {ndu[nd[0]], ndu[nd[1]], ndu[nd[2]], ndu[nd[3]]};
    const double cv[4] = {ndv[nd[0]], ndv[nd[1]], ndv[nd[2]], ndv[nd[3]]};
    const double4 w = reinterpret_cast<const double4*>(cnwt)[e];
    const double wt[4] = {w.x, w.y, w.z, w.w};
    sp_row(dencut, den[e], en[e], pre[e], vol[e], mass[e], wt, cu, cv, r);
  }
  block_flag_reduce(nflag, mine, r, nb, blockIdx.x, part);
}

// component rows by icpmat; a component's corners take its cell's cnwt and
// corner velocities (utils_kn_mxgathercncp, hydro_dr_print.f90:96-118)
__global__ void k_sp_components(MixArgs M, int nflag, double dencut,
                                const int32_t* __restrict__ ielnd,
                                const double* __restrict__ cnwt, const double* __restrict__ ndu,
                                const double* __restrict__ ndv, const int32_t* __restrict__ cpel,
                                int nb, int b0, double* __restrict__ part) {
  const int icp = blockIdx.x * blockDim.x + threadIdx.x;
  double r[kNq];
  int mine = -1;
  const int e = icp < M.ncp ? cpel[icp] : -1;
  if (e >= 0 && M.icpmat[icp] > 0) {
    mine = M.icpmat[icp] - 1;
    const int4 q = reinterpret_cast<const int4*>(ielnd)[e];
    const int nd[4] = {q.x - 1, q.y - 1, q.z - 1, q.w - 1};
    const double4 w = reinterpret_cast<const double4*>(cnwt)[e];
    const double wt[4] = {w.x, w.y, w.z, w.w};
    const double cu[4] = {ndu[nd[0]], ndu[nd[1]], ndu[nd[2]], ndu[nd[3]]};
    const double cv[4] = {ndv[nd[0]], ndv[nd[1]], ndv[nd[2]], ndv[nd[3]]};
    sp_row(dencut, M.cpdensity[icp], M.cpenergy[icp], M.cppressure[icp], M.cpvolume[icp],
           M.cpmass[icp], wt, cu, cv, r);
  }
  block_flag_reduce(nflag, mine, r, nb, b0 + blockIdx.x, part);
}

// element of each component, from the mixed-cell lists
__global__ void k_cp_element(MixArgs M, int32_t* __restrict__ cpel) {
  const int imx = blockIdx.x * blockDim.x + threadIdx.x;
  if (imx >= M.nmx) return;
  int icp = M.imxfcp[imx] - 1;
  for (int ii = 0; ii < M.imxncp[imx]; ++ii, ++icp) cpel[icp] = M.imxel[imx] - 1;
}

// sod() of check_kn_tests.f90:64-111
__device__ __forceinline__ void sod_exact(double xx, double time, double& r1, double& r2) {
  const double coeff = sqrt(1.4);
  r1 = -DBL_MAX; r2 = -DBL_MAX;
  if (xx <= -coeff * time) {
    r1 = 1.0; r2 = 2.5;
  } else if (xx <= -0.07027281256118326961 * time) {
    const double ss = xx / time;
    const double velocity = (5.0 / 6.0) * (ss + coeff);
    const double tt = ((velocity - ss) * (velocity - ss)) / 1.4;
    r1 = pow(tt, 2.5);
    r2 = r1 * tt / (0.4 * r1);
  } else if (xx <= 0.92745262004894994908 * time) {
    r1 = 0.42631942817849519385; r2 = 1.77760006942335264781;
  } else {
    if (time <= 28.53627624872492075028) {
      if (xx <= 1.75215573203017816370 * time) {
        r1 = 0.26557371170530706471; r2 = 2.85354088799095973738;
      } else {
        r1 = 0.125; r2 = 2.0;
      }
    } else if (time < 40.68191725689148697880) {
      if (xx <= (50.0 - (time - 28.53627624872492075028) * 1.01019363599101820444)) {
        r1 = 0.26557371170530706471; r2 = 2.85354088799095973738;
      } else {
        r1 = 0.50939531774381657731; r2 = 3.82996297061558546292;
      }
    }
  }
}

// check_kn_sod per element: (volume, |rho - rho_exact| V, |e - e_exact| V)
// at the centroid of geometry_kn_getcentroid (geometry_kn_centroid.f90:
// 29-55) of its corners (x, y)
__device__ __forceinline__ void l1_terms(const double x[4], const double y[4], double v, double den,
                                         double en, double x0, double scale, double t,
                                         double r[3]) {
  double cx = 0.0, rv = 0.0;
#pragma unroll
  for (int i1 = 0; i1 < 4; ++i1) {
    const int i2 = (i1 + 1) & 3;
    const double rr = x[i1] * y[i2] - x[i2] * y[i1];
    rv = rv + rr;
    cx = cx + rr * (x[i1] + x[i2]);
  }
  rv = 0.5 * rv;
  cx = (rv > 0.0) ? cx / (6.0 * rv) : 0.0;
  double s1, s2;
  sod_exact(scale * (cx - x0), scale * t, s1, s2);
  r[0] = v;
  r[1] = fabs(den - s1) * v;
  r[2] = fabs(en - s2) * v;
}

// the workgroup's three L1 sums into part[q * nb + b]; every thread of the
// workgroup must call it
__device__ __forceinline__ void block_l1_reduce(const double r[3], int nb, int b, double* part) {
  __shared__ double sh[kBlock / 64][3];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, t = threadIdx.x;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const double x = wave_fold(r[q], [](double a, double c) { return a + c; });
    if (lane == 63) sh[wid][q] = x;
  }
  __syncthreads();
  if (t < 3) {
    double x = sh[0][t];
    for (int w = 1; w < kBlock / 64; ++w) x = x + sh[w][t];
    part[(size_t)t * nb + b] = x;
  }
}

// the L1 sums from the corner arrays cnx, cny (4, nel) and the volume field
__global__ void __launch_bounds__(kBlock)
k_l1(int nel, const double* __restrict__ cnx, const double* __restrict__ cny,
     const double* __restrict__ vol, const double* __restrict__ den,
     const double* __restrict__ en, double x0, double scale, double time,
     double* __restrict__ part) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  double r[3] = {0.0, 0.0, 0.0};
  if (e < nel) {
    const double4 a = reinterpret_cast<const double4*>(cnx)[e];
    const double4 b = reinterpret_cast<const double4*>(cny)[e];
    const double x[4] = {a.x, a.y, a.z, a.w}, y[4] = {b.x, b.y, b.z, b.w};
    l1_terms(x, y, vol[e], den[e], en[e], x0, scale, time, r);
  }
  block_l1_reduce(r, gridDim.x, blockIdx.x, part);
}

// The record of a step in two launches, from the node set it wrote.  First
// every element's row and L1 terms (one gather of its nodes for both) into
// the workgroups' partials, and the record's place (counter[1], the next one
// in counter[0]); then one workgroup per column of the region table and one
// for the L1 pair, which write the record [nstep, time, region table
// (nreg x 9), L1 rho, L1 e] themselves.  res: a step on a tiling has its own
// outcome (its end is recorded by the next step); a step that did not
// complete leaves no record.  Sedov 512^2: 15 us a step, where a launch for
// the step's end and four for the record (one gather of the nodes for the
// rows, one for the L1 pair) took 33.
__device__ __forceinline__ bool no_record(const DevTimestep* ts, const DtResult* res) {
  return ts->skip || (res && (res->negvol | res->negvol2 | res->negvol3));
}

__global__ void __launch_bounds__(kBlock)
k_diag_elements(int nel, int nreg, double dencut, const int32_t* __restrict__ ielreg,
                const int32_t* __restrict__ ielnd, const double* __restrict__ den,
                const double* __restrict__ en, const double* __restrict__ pre,
                const double* __restrict__ mass, const double* __restrict__ ndx,
                const double* __restrict__ ndy, const double* __restrict__ ndu,
                const double* __restrict__ ndv, double x0, double scale,
                double* __restrict__ part, int32_t* __restrict__ counter, int maxrec,
                const DevTimestep* ts, const DtResult* res) {
  if (no_record(ts, res)) return;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    const int k = counter[0];
    counter[1] = k;
    if (k < maxrec) counter[0] = k + 1;
  }
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  double r[kNq], l[3] = {0.0, 0.0, 0.0};
  int mine = -1;
  if (e < nel) {
    const int4 q = reinterpret_cast<const int4*>(ielnd)[e];
    const int reg = ielreg[e];
    const double d = den[e], ee = en[e], p = pre[e], m = mass[e];
    const int nd[4] = {q.x - 1, q.y - 1, q.z - 1, q.w - 1};
    double x[4], y[4], cu[4], cv[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      x[c] = ndx[nd[c]];
      y[c] = ndy[nd[c]];
      cu[c] = ndu[nd[c]];
      cv[c] = ndv[nd[c]];
    }
    Iso g;
    sp_row_nodes(dencut, d, ee, p, m, x, y, cu, cv, g, r);
    if (reg > 0) mine = reg - 1;
    l1_terms(x, y, g.vol, d, ee, x0, scale, ts->time, l);
  }
  block_flag_reduce(nreg, mine, r, gridDim.x, blockIdx.x, part);
  block_l1_reduce(l, gridDim.x, blockIdx.x, part + (size_t)nreg * kNq * gridDim.x);
}

// one column of the per-workgroup partials (col[0, nb)) reduced by one
// workgroup: each thread combines b = t, t + kBlock, ... in order, then
// across the lanes and over the waves.  The result depends only on nb and
// the data.  Every thread of the workgroup must call it; all get the result.
__device__ __forceinline__ double column_reduce(int nb, int q, const double* __restrict__ col) {
  __shared__ double sh[kBlock / 64];
  const int t = threadIdx.x;
  double a = q_identity(q);
  // four loads in flight, combined in order
  int b = t;
  for (; b + 3 * kBlock < nb; b += 4 * kBlock) {
    const double v0 = col[b], v1 = col[b + kBlock], v2 = col[b + 2 * kBlock],
                 v3 = col[b + 3 * kBlock];
    a = q_combine(q, q_combine(q, q_combine(q, q_combine(q, a, v0), v1), v2), v3);
  }
  for (; b < nb; b += kBlock) a = q_combine(q, a, col[b]);
  a = wave_fold(a, [q](double x, double y) { return q_combine(q, x, y); });
  if ((t & 63) == 63) sh[t >> 6] = a;
  __syncthreads();
  double r = sh[0];
#pragma unroll
  for (int w = 1; w < kBlock / 64; ++w) r = q_combine(q, r, sh[w]);
  __syncthreads();
  return r;
}

// one workgroup per column i of an (nflag x kNq) table: out[i]
__global__ void __launch_bounds__(kBlock) k_flag_final(int nb, const double* __restrict__ part,
                                                       double* __restrict__ out) {
  const int i = blockIdx.x;
  const double r = column_reduce(nb, i % kNq, part + (size_t)i * nb);
  if (threadIdx.x == 0) out[i] = r;
}

// one workgroup: the three L1 sums
__global__ void __launch_bounds__(kBlock) k_l1_final(int nb, const double* __restrict__ part,
                                                     double* __restrict__ out) {
  for (int i = 0; i < 3; ++i) {
    const double r = column_reduce(nb, 0, part + (size_t)i * nb);
    if (threadIdx.x == 0) out[i] = r;
  }
}

// the record (k_diag_elements): workgroup c < nreg * kNq a column of the
// region table, the last one the L1 pair
__global__ void __launch_bounds__(kBlock)
k_diag_record(int nb, int nreg, const double* __restrict__ part, double* __restrict__ hist,
              const int32_t* __restrict__ counter, int maxrec, const DevTimestep* ts,
              const DtResult* res) {
  if (no_record(ts, res)) return;
  const int k = counter[1], c = blockIdx.x, nt = nreg * kNq;
  if (k >= maxrec) return;
  double* dst = hist + (size_t)k * (2 + nt + 2);
  if (c < nt) {
    const double r = column_reduce(nb, c % kNq, part + (size_t)c * nb);
    if (threadIdx.x == 0) dst[2 + c] = r;
    return;
  }
  double s[3];
  for (int i = 0; i < 3; ++i) s[i] = column_reduce(nb, 0, part + (size_t)(nt + i) * nb);
  if (threadIdx.x == 0) {
    dst[0] = (double)ts->nstep;
    dst[1] = ts->time;
    dst[2 + nt] = s[1] / s[0];
    dst[3 + nt] = s[2] / s[0];
  }
}

}  // namespace bl

using namespace bl;

namespace {

// the partials buffer, at least n doubles; a new buffer invalidates the
// captured step, whose diagnostics kernels hold the old one
double* diag_part(bl_handle_t* h, size_t n) {
  if (h->diag_part_n < n) {
    hipStreamSynchronize(h->stream);
    invalidate_graph(h);
    if (h->d_diag_part) hipFree(h->d_diag_part);
    h->d_diag_part = nullptr;
    h->diag_part_n = 0;
    if (hipMalloc(&h->d_diag_part, sizeof(double) * n) != hipSuccess) {
      set_error("out of device memory for diagnostics");
      return nullptr;
    }
    h->diag_part_n = n;
  }
  return h->d_diag_part;
}

// the final pass over nb workgroups' partials into dout (nflag rows on the
// device), then to out on the host
int final_to_host(bl_handle_t* h, int nflag, unsigned nb, const double* part, double* dout,
                  double* out) {
  hipLaunchKernelGGL(k_flag_final, dim3(nflag * kNq), dim3(kBlock), 0, h->stream, (int)nb, part,
                     dout);
  hipError_t e0 = hipGetLastError();
  hipError_t e1 = hipMemcpyAsync(out, dout, sizeof(double) * kNq * nflag,
                                 hipMemcpyDeviceToHost, h->stream);
  hipError_t e2 = hipStreamSynchronize(h->stream);
  if (e0 != hipSuccess || e1 != hipSuccess || e2 != hipSuccess) {
    set_error("diagnostics reduction failed");
    return BL_FAILURE;
  }
  return BL_SUCCESS;
}

}  // namespace

namespace bl {

// the per-step record of the fused step from the node set the step wrote
int launch_diag(Handle* h, const double* ndx, const double* ndy, const double* ndu,
                const double* ndv, const double* rho, const double* en, const double* pre,
                const DevTimestep* ts, const DtResult* res) {
  if (!h->diag_on) return BL_SUCCESS;
  if (!ts) ts = h->d_ts;
  if (!rho) rho = h->R(BL_ELDENSITY);
  if (!en) en = h->R(BL_ELENERGY);
  if (!pre) pre = h->R(BL_ELPRESSURE);
  const int nel = h->sz.nel, nreg = h->nreg;
  const unsigned nb = nblocks(nel);
  double* part = h->d_diag_part;  // sized by bl_set_diagnostics
  BL_LAUNCH(h, "diag_elements", k_diag_elements, nb, kBlock, nel, nreg, h->cfg.dencut,
            (const int32_t*)h->I(BL_IELREG), (const int32_t*)h->I(BL_IELND), rho, en, pre,
            (const double*)h->R(BL_ELMASS), ndx, ndy, ndu, ndv, h->diag_x0, h->diag_scale, part,
            h->d_diag_count, h->diag_max, ts, res);
  BL_LAUNCH(h, "diag_record", k_diag_record, nreg * kNq + 1, kBlock, (int)nb, nreg,
            (const double*)part, h->d_diag_hist, (const int32_t*)h->d_diag_count, h->diag_max, ts,
            res);
  return BL_SUCCESS;
}

}  // namespace bl

extern "C" {

int bl_shortprint(bl_handle_t* h, bl_flag_totals_t* region, bl_flag_totals_t* material) {
  bl_touch(h);
  if (!h || !region || !material) return BL_FAILURE;
  const int nel = h->sz.nel, nreg = h->sz.nreg, nmat = h->sz.nmat, ncp = h->sz.ncp;
  const unsigned nb = nblocks(nel), nbc = ncp > 0 ? nblocks(ncp) : 0;
  const int nf = std::max(std::max(nreg, nmat), 1);
  const size_t used = (size_t)(nb + nbc) * nf * kNq;
  double* part = diag_part(h, used + (size_t)nf * kNq);
  if (!part) return BL_FAILURE;
  double* dout = part + used;
  BL_LAUNCH(h, "shortprint", k_sp_elements, nb, kBlock, nel, nreg, h->cfg.dencut,
            (const int32_t*)h->I(BL_IELREG), (const int32_t*)h->I(BL_IELND),
            (const double*)h->R(BL_ELDENSITY), (const double*)h->R(BL_ELENERGY),
            (const double*)h->R(BL_ELPRESSURE), (const double*)h->R(BL_ELVOLUME),
            (const double*)h->R(BL_ELMASS), (const double*)h->R(BL_CNWT),
            (const double*)h->R(BL_NDU), (const double*)h->R(BL_NDV), (int)nb, part);
  if (final_to_host(h, nreg, nb, part, dout, reinterpret_cast<double*>(region)))
    return BL_FAILURE;
  BL_LAUNCH(h, "shortprint", k_sp_elements, nb, kBlock, nel, nmat, h->cfg.dencut,
            (const int32_t*)h->I(BL_IELMAT), (const int32_t*)h->I(BL_IELND),
            (const double*)h->R(BL_ELDENSITY), (const double*)h->R(BL_ELENERGY),
            (const double*)h->R(BL_ELPRESSURE), (const double*)h->R(BL_ELVOLUME),
            (const double*)h->R(BL_ELMASS), (const double*)h->R(BL_CNWT),
            (const double*)h->R(BL_NDU), (const double*)h->R(BL_NDV), (int)(nb + nbc), part);
  if (ncp > 0) {
    int32_t* cpel = nullptr;
    BL_HIP(hipMalloc(&cpel, sizeof(int32_t) * ncp));
    // -1: a component in no mixed cell's range is left out
    BL_HIP(hipMemsetAsync(cpel, 0xff, sizeof(int32_t) * ncp, h->stream));
    MixArgs M = make_mix(h);
    hipLaunchKernelGGL(k_cp_element, dim3(nblocks(h->sz.nmx)), dim3(kBlock), 0, h->stream, M,
                       cpel);
    // the components' workgroups follow the elements': the final pass adds
    // both, as the reference's second call adds to the first's rows
    hipLaunchKernelGGL(k_sp_components, dim3(nbc), dim3(kBlock), 0, h->stream, M, nmat,
                       h->cfg.dencut, (const int32_t*)h->I(BL_IELND),
                       (const double*)h->R(BL_CNWT), (const double*)h->R(BL_NDU),
                       (const double*)h->R(BL_NDV), (const int32_t*)cpel, (int)(nb + nbc), (int)nb,
                       part);
    hipError_t e = hipGetLastError();
    hipStreamSynchronize(h->stream);
    hipFree(cpel);
    if (e != hipSuccess) { set_error("shortprint components failed"); return BL_FAILURE; }
  }
  return final_to_host(h, nmat, nb + nbc, part, dout, reinterpret_cast<double*>(material));
}

int bl_sod_l1(bl_handle_t* h, double time, double x0, double scale, double* l1) {
  bl_touch(h);
  if (!h || !l1) return BL_FAILURE;
  const int nel = h->sz.nel;
  const unsigned nb = nblocks(nel);
  double* part = diag_part(h, (size_t)(nb + 1) * 3);
  if (!part) return BL_FAILURE;
  BL_LAUNCH(h, "sod_l1", k_l1, nb, kBlock, nel, (const double*)h->R(BL_CNX),
            (const double*)h->R(BL_CNY), (const double*)h->R(BL_ELVOLUME),
            (const double*)h->R(BL_ELDENSITY), (const double*)h->R(BL_ELENERGY), x0, scale, time,
            part);
  double s[3], *dout = part + 3 * (size_t)nb;
  BL_LAUNCH(h, "sod_l1", k_l1_final, 1, kBlock, (int)nb, (const double*)part, dout);
  BL_HIP(hipMemcpyAsync(s, dout, sizeof(s), hipMemcpyDeviceToHost, h->stream));
  BL_HIP(hipStreamSynchronize(h->stream));
  l1[0] = s[1] / s[0];
  l1[1] = s[2] / s[0];
  return BL_SUCCESS;
}

int bl_set_diagnostics(bl_handle_t* h, int32_t on, double x0, double scale, int32_t maxrec) {
  bl_touch(h);
  if (!h) return BL_FAILURE;
  BL_HIP(hipStreamSynchronize(h->stream));
  invalidate_graph(h);
  h->diag_on = false;
  if (!on) return BL_SUCCESS;
  if (maxrec <= 0 || h->nreg <= 0) {
    set_error("bl_set_diagnostics: maxrec and the region count must be positive");
    return BL_FAILURE;
  }
  const int nreg = h->nreg;
  const unsigned nb = nblocks(h->sz.nel);
  if (!diag_part(h, (size_t)nb * ((size_t)nreg * kNq + 3))) return BL_FAILURE;
  if (h->d_diag_hist) hipFree(h->d_diag_hist);
  h->d_diag_hist = nullptr;
  const size_t rec = 2 + kNq * (size_t)nreg + 2;
  BL_HIP(hipMalloc(&h->d_diag_hist, sizeof(double) * rec * maxrec));
  if (!h->d_diag_count) BL_HIP(hipMalloc(&h->d_diag_count, 2 * sizeof(int32_t)));
  BL_HIP(hipMemsetAsync(h->d_diag_count, 0, 2 * sizeof(int32_t), h->stream));
  BL_HIP(hipStreamSynchronize(h->stream));
  h->diag_on = true;
  h->diag_x0 = x0;
  h->diag_scale = scale;
  h->diag_max = maxrec;
  return BL_SUCCESS;
}

int bl_diagnostics(bl_handle_t* h, int32_t maxrec, double* out, int32_t* nrec) {
  bl_touch(h);
  if (!h || !nrec) return BL_FAILURE;
  *nrec = 0;
  if (!h->d_diag_count || !h->d_diag_hist) return BL_SUCCESS;
  int32_t n = 0;
  BL_HIP(hipMemcpyAsync(&n, h->d_diag_count, sizeof(int32_t), hipMemcpyDeviceToHost, h->stream));
  BL_HIP(hipStreamSynchronize(h->stream));
  n = std::min(n, std::min(maxrec, h->diag_max));
  const size_t rec = 2 + kNq * (size_t)h->nreg + 2;
  if (n > 0 && out)
    BL_HIP(hipMemcpy(out, h->d_diag_hist, sizeof(double) * rec * n, hipMemcpyDeviceToHost));
  *nrec = n;
  return BL_SUCCESS;
}

}  // extern "C"
