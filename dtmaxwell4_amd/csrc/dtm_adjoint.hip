// dtm_adjoint.hip — device side of the design-gradient adjoint.
//
// Objective: J = sum_m |F_m|^2, F_m = sum_{n=0}^{N-1} Ez_m^{n+1} e^{i w (n+1) dt} dt
// over monitor cells m (the running DFT of the probes), differentiated with
// respect to the inverse permittivity of the design box.
//
// The leapfrog step (H^{n+1/2} = H^{n-1/2} - dt Ce E^n, E^{n+1} = E^n + dt M Ch
// H^{n+1/2}, M = 1/eps, Ch = Ce^T for the (2,4) staggered differences) has
// the transposed step
//   lH~ = lH + dt Ce (M lE^{n+1}),   lE^n = lE^{n+1} - dt Ch lH~ + dJ/dE^n,
// which in zeta = M lE and eta = -lH~ is the forward step itself:
//   eta -= dt Ce zeta,   zeta += dt M Ch eta + M dJ/dE^n.
// So the adjoint runs the forward sweeps backward in n on (zeta, eta), with
// the objective's derivative injected at the monitors, and
//   dJ/dM_c = sum_n lE_c^{n+1} dt (Ch H^{n+1/2})_c = sum_n eps_c^2 zeta_c^{n+1} (E_c^{n+1} - E_c^n)
// from the design-box E history of the forward run.  (The CPML is applied in
// its forward form to the adjoint fields, an absorbing layer for them too;
// the reference has no adjoint.)
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdio.h>

#include <algorithm>

#include "dtm_internal.h"

namespace dtm {

namespace {

// The design cells and the monitors of some x planes: cells [b0, b1) of the
// box, monitors whose cell index lies in [q0, q1).
struct Part {
  long long b0, b1, q0, q1;
};
__device__ __forceinline__ long long design_cell(const Grid& g, const Materials& mt, long long b) {
  const int k = mt.d_k0 + (int)(b % mt.d_nk);
  const int j = mt.d_j0 + (int)((b / mt.d_nk) % mt.d_nj);
  const int i = mt.d_i0 + (int)(b / ((long long)mt.d_nk * mt.d_nj));
  return i * g.sx + j * g.sy + k;
}

// The first nbs blocks: E of the design box, three components, into
// out[c * nd + cell]; the rest: series[m] = Ez at the monitor cells.
__global__ __launch_bounds__(256) void k_adj_record(Grid g, Fields<0> f, Materials mt, Part pt, float* out, unsigned nbs,
                                                    const long long* q, int nmon, float* series) {
  if (blockIdx.x < nbs) {
    const long long b = pt.b0 + blockIdx.x * 256LL + threadIdx.x;
    if (b >= pt.b1) return;
    const long long nd = (long long)mt.d_ni * mt.d_nj * mt.d_nk, cell = design_cell(g, mt, b);
    for (int c = 0; c < 3; c++) out[c * nd + b] = f.E[c][cell];
    return;
  }
  const int m = (blockIdx.x - nbs) * 256 + threadIdx.x;
  if (m < nmon && q[m] >= pt.q0 && q[m] < pt.q1) series[m] = f.E[2][q[m]];
}

// The first nbg blocks: acc[cell] += sum_c eps^2 zeta_c (E1_c - E0_c) (design
// inverse permittivity is isotropic); the rest: zeta_z += M dJ/dEz^n at the
// monitors, dJ/dEz_m^n = 2 dt Re(conj(F_m) e^{i w n dt}).  Both at once only when
// no monitor lies in the design box, so the two touch disjoint cells.
__global__ __launch_bounds__(256) void k_adj_inject_grad(Grid g, Fields<0> f, Materials mt, Part pt, const float* e0,
                                                         const float* e1, double* acc, unsigned nbg,
                                                         const long long* q, const float* inv_eps, const double* F,
                                                         int nmon, double w, double dt, long long n) {
  if (blockIdx.x < nbg) {
    const long long b = pt.b0 + blockIdx.x * 256LL + threadIdx.x;
    if (b >= pt.b1) return;
    const long long nd = (long long)mt.d_ni * mt.d_nj * mt.d_nk, qq = design_cell(g, mt, b);
    const double eps = 1.0 / (double)mt.d_inv_eps[b];
    double sum = 0.0;
    for (int c = 0; c < 3; c++) sum += (double)f.E[c][qq] * ((double)e1[c * nd + b] - (double)e0[c * nd + b]);
    acc[b] += eps * eps * sum;
    return;
  }
  const int m = (blockIdx.x - nbg) * 256 + threadIdx.x;
  if (m >= nmon || q[m] < pt.q0 || q[m] >= pt.q1) return;
  double sn, cn;
  sincos(w * (double)n * dt, &sn, &cn);
  const double gJ = 2.0 * dt * (F[2 * m] * cn + F[2 * m + 1] * sn);
  f.E[2][q[m]] += (float)(gJ * inv_eps[m]);
}

void check(const char* what) { note_launch(what); }

unsigned blocks_for(long long n) { return n > 0 ? (unsigned)((n + 255) / 256) : 0u; }

Part part(const Grid& g, const Materials& mt, int i0, int i1) {
  const long long pl = (long long)mt.d_nj * mt.d_nk;
  return Part{pl * std::min(std::max(0, i0 - mt.d_i0), mt.d_ni), pl * std::max(0, std::min(mt.d_ni, i1 - mt.d_i0)),
              g.sx * i0, g.sx * i1};
}

}  // namespace

void launch_adj_record(const Grid& g, const void* fields, const Materials& mt, int i0, int i1, float* snap,
                       const long long* q, int nmon, float* series, hipStream_t st) {
  const Part p = part(g, mt, i0, i1);
  const unsigned nbs = snap ? blocks_for(p.b1 - p.b0) : 0, nbm = series ? blocks_for(nmon) : 0;
  if (nbs + nbm == 0) return;
  hipLaunchKernelGGL(k_adj_record, dim3(nbs + nbm), dim3(256), 0, st, g, *static_cast<const Fields<0>*>(fields), mt, p,
                     snap, nbs, q, nmon, series);
  check("k_adj_record");
}

void launch_adj_inject_grad(const Grid& g, const void* fields, const Materials& mt, int i0, int i1, const float* e0,
                            const float* e1, double* acc, const long long* q, const float* inv_eps, const double* F,
                            int nmon, double w, double dt, long long n, hipStream_t st) {
  const Part p = part(g, mt, i0, i1);
  const unsigned nbg = e0 ? blocks_for(p.b1 - p.b0) : 0, nbm = q ? blocks_for(nmon) : 0;
  if (nbg + nbm == 0) return;
  hipLaunchKernelGGL(k_adj_inject_grad, dim3(nbg + nbm), dim3(256), 0, st, g, *static_cast<const Fields<0>*>(fields),
                     mt, p, e0, e1, acc, nbg, q, inv_eps, F, nmon, w, dt, n);
  check("k_adj_inject_grad");
}

}  // namespace dtm
