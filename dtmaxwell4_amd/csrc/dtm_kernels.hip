// dtm_kernels.hip — the kernels around the half-step sweeps (dtm_sweep.hip):
// TF/SF corrections and their tables, dispersive and gyrotropic cells, soft
// sources, probes, and conversion of half-precision fields.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdio.h>

#include <algorithm>

#include "dtm_box.h"
#include "dtm_internal.h"
#include "dtm_probe.h"

namespace dtm {

// ------------------------------------------------------- storage helpers
__device__ __forceinline__ float ld(const float* F, long long q, float) { return F[q]; }
__device__ __forceinline__ float ld(const __half* F, long long q, float inv) {
  return __half2float(F[q]) * inv;
}
__device__ __forceinline__ void st(float* F, long long q, float v, float) { F[q] = v; }
__device__ __forceinline__ void st(__half* F, long long q, float v, float s) {
  F[q] = __float2half_rn(v * s);
}
// one cell of component comp (Ex .. Hz = 0 .. 5) with the FP32 zone: xq is
// the cell's zone index (exact_idx) or -1; the half array always holds the
// rounded zone value, so readers that ignore the zone see FP16 precision
__device__ __forceinline__ float ldx(const float* F, long long q, float inv, const Exact&, int, int) {
  return ld(F, q, inv);
}
__device__ __forceinline__ float ldx(const __half* F, long long q, float inv, const Exact& xz, int comp, int xq) {
  return xq >= 0 ? xz.f[comp][xq] : ld(F, q, inv);
}
__device__ __forceinline__ void stx(float* F, long long q, float v, float s, const Exact&, int, int) {
  st(F, q, v, s);
}
__device__ __forceinline__ void stx(__half* F, long long q, float v, float s, const Exact& xz, int comp, int xq) {
  if (xq >= 0) xz.f[comp][xq] = v;
  st(F, q, v, s);
}

// Neighbour index along one axis with the boundary rule: -1 => zero field.
__device__ __forceinline__ int nbr(int v, int o, int n, int per) {
  int w = v + o;
  if (w >= 0 && w < n) return w;
  if (!per) return -1;
  return w < 0 ? w + n : w - n;
}


// ------------------------------------------------------- incident fields
__device__ __forceinline__ void wave3(int waveform, double p, double w, double kEnv, double t0, double tw,
                      double& f0, double& f1, double& f2) {
  if (waveform == 0) {  // raised-cosine window (signal.hpp:71-77)
    const double kp = p * kEnv;
    if (kp < 0.0 || kp > 2.0 * M_PI) {
      f0 = f1 = f2 = 0.0;
      return;
    }
    double sp, cp, sk, ck;
    sincos(p, &sp, &cp);
    sincos(kp, &sk, &ck);
    f0 = sp * 0.5 * (1.0 - ck);
    f1 = 0.5 * cp * (1.0 - ck) + 0.5 * kEnv * sp * sk;
    f2 = -0.5 * sp * (1.0 - ck) + kEnv * cp * sk + 0.5 * kEnv * kEnv * sp * ck;
  } else {  // Gaussian-modulated sine, or the bare Gaussian (waveform 2, signal.hpp:55-57)
    const double a = 1.0 / (w * tw);
    const double u = (p / w - t0) / tw;
    const double g = exp(-u * u);
    const double g1 = -2.0 * u * a * g;
    const double g2 = (4.0 * u * u * a * a - 2.0 * a * a) * g;
    if (waveform == 2) {
      f0 = g;
      f1 = g1;
      f2 = g2;
      return;
    }
    double sp, cp;
    sincos(p, &sp, &cp);
    f0 = g * sp;
    f1 = g1 * sp + g * cp;
    f2 = g2 * sp + 2.0 * g1 * cp - g * sp;
  }
}

// Incident value of component comp (0..5) at half-coordinates h, time t.
// Dipole: signal.hpp:58-96; plane wave: signal.hpp:17-49.
__device__ __forceinline__ double incident(const Tfsf& s, int comp, int hx, int hy, int hz, double t) {
  const double x = hx * s.half_d[0], y = hy * s.half_d[1], z = hz * s.half_d[2];
  if (s.kind == 1) {
    double n0 = x - s.dip[0], n1 = y - s.dip[1], n2 = z - s.dip[2];
    const double R = sqrt(n0 * n0 + n1 * n1 + n2 * n2);
    const double c = s.cSrc, w = s.w;
    double f0, f1, f2;
    wave3(s.waveform, w * t - w / c * R, w, s.kEnv, s.t0, s.tw, f0, f1, f2);
    const double d = s.amp * f0, ds = s.amp * w * f1, dss = s.amp * w * w * f2;
    n0 /= R;
    n1 /= R;
    n2 /= R;
    // dipole along the unit axis u (theta, phi; theta = 0: the reference's z
    // dipole, signal.hpp:70-72): d = d u, so (dss x n) x n = dss ((u.n) n - u)
    const double u0 = s.st * s.cph, u1 = s.st * s.sph, u2 = s.ct;
    const double un = u0 * n0 + u1 * n1 + u2 * n2;
    if (comp < 3) {
      const double nc = comp == 0 ? n0 : (comp == 1 ? n1 : n2);
      const double uc = comp == 0 ? u0 : (comp == 1 ? u1 : u2);
      const double t2 = dss * (un * nc - uc);
      return c * (t2 / (c * c * R) + (3.0 * ds * un * nc - ds * uc) / (c * R * R) +
                  (3.0 * d * un * nc - d * uc) / (R * R * R));
    } else {
      // (v u) x n = v (u1 n2 - u2 n1, u2 n0 - u0 n2, u0 n1 - u1 n0)
      const int a = comp - 3;
      const double cz = a == 0 ? u1 * n2 - u2 * n1 : (a == 1 ? u2 * n0 - u0 * n2 : u0 * n1 - u1 * n0);
      return dss * cz / (c * c * R) + ds * cz / (c * R * R);
    }
  } else {
    const double phase = s.w * t - s.kx * (x - s.pos[0]) - s.ky * (y - s.pos[1]) - s.kz * (z - s.pos[2]);
    double f0, f1, f2;
    wave3(s.waveform, phase, s.w, s.kEnv, s.t0, s.tw, f0, f1, f2);
    const double sv = s.amp * f0;
    const double Ephi = s.Imp * sv * s.cps, Eth = s.Imp * sv * s.sps;
    const double Hth = -sv * s.cps, Hphi = sv * s.sps;
    switch (comp) {
      case 0: return -Ephi * s.sph + Eth * s.ct * s.cph;
      case 1: return Ephi * s.cph + Eth * s.ct * s.sph;
      case 2: return -Eth * s.st;
      case 3: return -Hphi * s.sph + Hth * s.ct * s.cph;
      case 4: return Hphi * s.cph + Hth * s.ct * s.sph;
      default: return -Hth * s.st;
    }
  }
}


// Sum over the 4 stencil neighbours along axis a, which hold component cq, of
// the TF/SF corrections (genAlg.py:219-221) weighted by (+1,-27,+27,-1).
// The neighbours differ from the point only along a, so no face is crossed
// unless the point lies inside the box on the other two axes; then a
// neighbour crosses when its a-coordinate is on the other side of [hlo, hhi].
__device__ __forceinline__ float tfsf_dcorr(const Tfsf& s, int hx, int hy, int hz, int a, int cq, double t) {
  const bool inx = hx >= s.hlo[0] && hx <= s.hhi[0], iny = hy >= s.hlo[1] && hy <= s.hhi[1],
             inz = hz >= s.hlo[2] && hz <= s.hhi[2];
  if (!((a == 0 || inx) && (a == 1 || iny) && (a == 2 || inz))) return 0.f;
  const int h = a == 0 ? hx : (a == 1 ? hy : hz), lo = s.hlo[a], hi = s.hhi[a];
  const bool pin = a == 0 ? inx : (a == 1 ? iny : inz);
  double acc = 0.0;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int hq = h + 2 * q - 3;
    const bool qin = hq >= lo && hq <= hi;
    if (qin == pin) continue;
    const bool qsf = s.sf_inside ? qin : !qin;  // the neighbour is in the scattered-field region
    const double v = incident(s, cq, a == 0 ? hq : hx, a == 1 ? hq : hy, a == 2 ? hq : hz, t);
    const double wt = q == 0 ? 1.0 : (q == 1 ? -27.0 : (q == 2 ? 27.0 : -1.0));
    acc += wt * (qsf ? v : -v);
  }
  return (float)acc;
}

// -------------------------------------------------------- CPML helpers
__device__ __forceinline__ int slab_index(int v, int n, int plo, int phi) {
  if (v < plo) return v;
  if (v >= n - phi) return plo + v - (n - phi);
  return -1;
}

__device__ __forceinline__ long long psi_index(const Grid& g, const Cpml& p, int a, int s, int i, int j,
                                               int k) {
  const int P = p.plo[a] + p.phi[a];
  if (a == 0) return ((long long)s * g.ny + j) * g.nz + k;
  if (a == 1) return ((long long)i * P + s) * g.nz + k;
  return ((long long)i * g.ny + j) * P + s;
}

// ============================================================ ADE cells
// Dispersive / gyrotropic cells: countDisp (dispersion.cpp:85-99) and the
// magnetised-plasma current, from the curl H the E sweep stored.
//
// One lane per cell of the bounding box (dtm_box.h).  A box of a
// few 10^5 cells is bound by its chain of loads more than by its bytes: the
// special classes are a mask in the arguments, so a cell's class byte says at
// once whether its state is needed, all of that is loaded together (NP and
// GYRO say which arrays there are, so that nothing branches), and the
// coefficients are scalar loads, one pass per distinct class of the wave.
// A Drude + Lorentz sphere of radius 40 (531441 cells in its box): FP32 15.7 us,
// FP16 with the FP32 zone 18.9, against 20.7 and 30 with the class entry, the
// material and each pole fetched in turn by the lane that needs them.
template <int STORE> struct AdeArgs {
  BoxUnits un;
  int ni, nj, nk, i0, j0, k0;  // the box
  long long sx, sy;
  const uint8_t* cls;
  decltype(Fields<STORE>::E) E, Ed;  // E^n, E^{n+1}
  float *curl[3], *Em[3], *Jg[3], *Jp[3][kMaxPoles], *Jm[3][kMaxPoles];
  float ie[3], se[3], dt;
  const ClassEntry* table;
  const AdeMat* mats;
  const GyroMat* gmats;
  int wide;                             // more than 32 classes
  unsigned special[kMaxClasses / 32];   // the classes of dispersive and gyrotropic cells, one bit each
  int d_on, d0[3], dn[3];  // design box
  Exact xz;
};
template <int STORE, int NP, bool GYRO, bool XZ>
__global__ __launch_bounds__(kBoxBlock) void k_ade(AdeArgs<STORE> A) {
  const unsigned long long pl = (unsigned long long)(unsigned)A.nj * (unsigned)A.nk;  // cells of a plane of the box
  unsigned ip;
  unsigned long long loc;
  const bool live = box_lane(A.un, (unsigned)A.ni, pl, blockIdx.x, threadIdx.x, ip, loc);
  const int jb = pl >> 32 ? (int)(loc / (unsigned)A.nk) : (int)((unsigned)loc / (unsigned)A.nk);
  const int i = A.i0 + (int)ip, j = A.j0 + jb;
  const int k = A.k0 + (int)(loc - (unsigned long long)jb * (unsigned)A.nk);
  const long long q = i * A.sx + j * A.sy + k;
  const unsigned long long b = ip * pl + loc;
  using U4 = unsigned __attribute__((ext_vector_type(4)));
  using TableK = __attribute__((address_space(4))) const U4;  // ClassEntry: inv_eps, then mat and special bytes
  using AdeK = __attribute__((address_space(4))) const AdeMat;
  using GyroK = __attribute__((address_space(4))) const GyroMat;
  unsigned cls = 0;
  float En[3], curl[3], Em[3], Jp[3][NP + 1], Jm[3][NP + 1], J0[3];
  bool mine = false;  // a cell of the box that this kernel updates
  int xq = -1;
  if (live) {
    if (A.cls) cls = A.cls[q];
    unsigned word = A.special[0];
    if (A.wide) {
#pragma unroll
      for (int w = 1; w < kMaxClasses / 32; w++) word = cls >> 5 == w ? A.special[w] : word;
    }
    mine = (word >> (cls & 31)) & 1u;
    if (A.d_on) {
      const int di = i - A.d0[0], dj = j - A.d0[1], dk = k - A.d0[2];
      if (di >= 0 && di < A.dn[0] && dj >= 0 && dj < A.dn[1] && dk >= 0 && dk < A.dn[2]) mine = false;
    }
  }
  if (mine) {
#pragma unroll
    for (int c = 0; c < 3; c++) {
      En[c] = ld(A.E[c], q, A.ie[c]);
      curl[c] = A.curl[c][b];
      Em[c] = A.Em[c][b];
#pragma unroll
      for (int p = 0; p < NP; p++) {
        Jp[c][p] = A.Jp[c][p][b];
        Jm[c][p] = A.Jm[c][p][b];
      }
      if (GYRO) J0[c] = A.Jg[c][b];
    }
    if (XZ) {
      xq = exact_idx(A.xz, i, j, k);
      if (xq >= 0)
#pragma unroll
        for (int c = 0; c < 3; c++) En[c] = A.xz.f[c][xq];
    }
  }
  auto put = [&](int c, float v) {
    if (XZ && xq >= 0) A.xz.f[c][xq] = v;
    st(A.Ed[c], q, v, A.se[c]);
  };
  for (unsigned long long todo = __builtin_amdgcn_ballot_w64(mine); todo != 0;) {
    const unsigned id = __builtin_amdgcn_readlane(cls, __builtin_ctzll(todo));
    const bool now = mine && cls == id;
    todo &= ~__builtin_amdgcn_ballot_w64(now);
    const U4 ce = ((TableK*)A.table)[id];
    const unsigned special = ce[3] >> 24;
    if (!now) continue;
    if (GYRO && (special & 8)) {
      GyroK& gm = ((GyroK*)A.gmats)[ce[3] & 0xff];
#pragma unroll
      for (int r = 0; r < 3; r++) {
        float v = 0.f;
#pragma unroll
        for (int t = 0; t < 3; t++) v += __builtin_fmaf(gm.A[3 * r + t], J0[t], gm.B[3 * r + t] * En[t]);
        A.Jg[r][b] = v;
        curl[r] -= v;
      }
    }
#pragma unroll
    for (int c = 0; c < 3; c++) {
      if (special & (1u << c)) {
        AdeK& am = ((AdeK*)A.mats)[(ce[3] >> (8 * c)) & 0xff];
        const int np = am.np;
        float kE[3], kEJ[NP + 1][2], kJ[NP + 1][5];
#pragma unroll
        for (int t = 0; t < 3; t++) kE[t] = am.kE[t];
#pragma unroll
        for (int p = 0; p < NP; p++) {
          kEJ[p][0] = am.kEJ[p][0];
          kEJ[p][1] = am.kEJ[p][1];
#pragma unroll
          for (int t = 0; t < 5; t++) kJ[p][t] = am.kJ[p][t];
        }
        const float Ep = En[c], em = Em[c];
        const float rotdt = A.dt * curl[c];
        float sum = 0.f;
#pragma unroll
        for (int p = 0; p < NP; p++)
          if (p < np) sum += __builtin_fmaf(kEJ[p][0], Jp[c][p], kEJ[p][1] * Jm[c][p]);
        const float Enew = __builtin_fmaf(kE[2], rotdt, __builtin_fmaf(kE[0], em, kE[1] * Ep)) - sum;
#pragma unroll
        for (int p = 0; p < NP; p++)
          if (p < np) {
            const float jp = Jp[c][p];
            float jn = __builtin_fmaf(kJ[p][0], jp, kJ[p][1] * Jm[c][p]);
            jn = __builtin_fmaf(kJ[p][2], Enew, jn);
            jn = __builtin_fmaf(kJ[p][3], em, jn);
            A.Jm[c][p][b] = jp;
            A.Jp[c][p][b] = __builtin_fmaf(kJ[p][4], Ep, jn);
          }
        A.Em[c][b] = Ep;
        put(c, Enew);
      } else {
        put(c, __builtin_fmaf(A.dt * __uint_as_float(ce[c]), curl[c], En[c]));
      }
    }
  }
}

// ====================================================== TF/SF correction
// For a cell in the face band of axis a, the two components with a
// derivative along a get the TF/SF term of genAlg.py:219-221 added to their
// stencil sum.  The sweep is linear in that sum, so the correction is
//   H_c -= dt * s * (1 + c_pml) * D,   psi += c_pml * D      (H half)
//   E_c += dt * ie * s * (1 + c_pml) * D, psi += c_pml * D   (E half)
// with s = +1 for the first curl term and -1 for the second; a dispersive
// component gets C3 * s * (1+c_pml) * D and its J^{n+1} the matching
// kJ2 * dE (dispersion.cpp:84-99 is linear in the curl).
// MODE 2 (H pre-correction before a fused step, on H^{n-1/2}): the fused
// step's own psi update then carries c*D, so psi gets c*D/b and H gets
// -dt*s*D only.
// One thread per cell of the union of the face bands: the cell belongs to
// the first band that contains it, and that thread applies the terms of
// every axis whose band holds the cell, so cells where bands of different
// axes overlap (box edges and corners) are written by one thread only.
// Cell and band of a thread: 32-bit arithmetic (band cells number far fewer
// than 2^31; 64-bit division would dominate the kernel).  Each band starts at
// a multiple of 64 threads, so a wavefront lies in one band: the band index is
// found from the wavefront's first thread and the band tables are read with
// scalar loads.  False: padding of a band, or the cell of an earlier band.
__device__ __forceinline__ bool band_has(const TfsfBands& bands, int r, int q, int i, int j, int k) {
  const Region& Q = bands.r[q];  // (only bands that overlap band r can hold a cell of it)
  return ((bands.ovl[r] >> q) & 1u) && i >= Q.i0 && i < Q.i1 && j >= Q.j0 && j < Q.j1 && k >= Q.k0 && k < Q.k1;
}
__device__ __forceinline__ bool band_cell(const TfsfBands& bands, int& r, int& i, int& j, int& k) {
  const unsigned gid = blockIdx.x * blockDim.x + threadIdx.x;
  const unsigned g0 = __builtin_amdgcn_readfirstlane(gid);
  r = 0;
  while (r < bands.n && g0 >= bands.start[r + 1]) r++;
  if (r >= bands.n) return false;
  const Region& R = bands.r[r];
  const unsigned nk = (unsigned)(R.k1 - R.k0), nj = (unsigned)(R.j1 - R.j0);
  unsigned loc = gid - bands.start[r];
  if (loc >= nk * nj * (unsigned)(R.i1 - R.i0)) return false;
  const unsigned lk = loc % nk;
  loc /= nk;
  k = R.k0 + (int)lk;
  j = R.j0 + (int)(loc % nj);
  i = R.i0 + (int)(loc / nj);
  for (int r2 = 0; r2 < r; r2++)
    if (band_has(bands, r, r2, i, j, k)) return false;
  return true;
}

// The correction D of the derivative along axis a in curl component c (t 0:
// its first term, 1: its second), through the layer: into dc, the curl
// correction per component, and dc2, its part on the stored split-field part.
template <int MODE>
__device__ __forceinline__ void tfsf_term(const Grid& g, const Cpml& pm, int a, int c, int t, float D, int i, int j,
                                          int k, float* dc, float* dc2) {
  constexpr int HALF = MODE == 1 ? 1 : 0;
  auto pos = [&](int ax) { return ax == 0 ? i : (ax == 1 ? j : k); };
  auto add = [&](float* d, float v) {
#pragma unroll
    for (int e = 0; e < 3; e++)
      if (e == c) d[e] += v;
  };
  const float sgn = t == 0 ? 1.0f : -1.0f;
  const int slot = t == 0 ? 1 : 0;  // psi slots 1 and 0 of axis a
  float cp = 0.0f;
  if (pm.on && pm.split) {  // split-field layer: the part of axis a gets k2 * D
    auto k2_of = [&](int ax) {  // 1 off the slab of axis ax
      const int n = ax == 0 ? g.nx : (ax == 1 ? g.ny : g.nz);
      if (slab_index(pos(ax), n, pm.plo[ax], pm.phi[ax]) < 0) return 1.0f;
      return HALF == 0 ? pm.cH[ax][pos(ax)] : pm.cE[ax][pos(ax)];
    };
    const float k2 = k2_of(a);
    // the cell keeps split parts when either curl axis has k2 != 1; the
    // second curl axis (t = 1) owns the stored part
    if (k2 != 1.0f || k2_of(t == 0 ? (c + 2) % 3 : (c + 1) % 3) != 1.0f) {
      add(dc, sgn * k2 * D);
      if (t == 1) add(dc2, sgn * k2 * D);
      return;
    }
  } else if (pm.on) {
    const int n = a == 0 ? g.nx : (a == 1 ? g.ny : g.nz);
    const int si = slab_index(pos(a), n, pm.plo[a], pm.phi[a]);
    if (si >= 0) {
      cp = HALF == 0 ? pm.cH[a][pos(a)] : pm.cE[a][pos(a)];
      float* psi = HALF == 0 ? pm.psiH[a][slot] : pm.psiE[a][slot];
      const long long pq = psi_index(g, pm, a, si, i, j, k);
      if (MODE == 2) {
        psi[pq] += cp * D / pm.bH[a][pos(a)];
        cp = 0.0f;
      } else {
        psi[pq] += cp * D;
      }
    }
  }
  add(dc, sgn * (1.0f + cp) * D);
}

// Adds the corrections of a cell to its fields.
template <int STORE, int MODE>
__device__ __forceinline__ void tfsf_apply(const Grid& g, const Fields<STORE>& f, const Scales& sc, const Cpml& pm,
                                           const Materials& mt, const Ade& ade, int i, int j, int k, const float* dc,
                                           const float* dc2) {
  const long long q = i * g.sx + j * g.sy + k;
  const int xq = STORE == 1 ? exact_idx(sc.xz, i, j, k) : -1;
  if (MODE != 1) {
#pragma unroll
    for (int c = 0; c < 3; c++) {
      if (dc[c] != 0.0f)
        stx(f.H[c], q, ldx(f.H[c], q, sc.ih[c], sc.xz, 3 + c, xq) - g.dt * dc[c], sc.sh[c], sc.xz, 3 + c, xq);
      if (dc2[c] != 0.0f) pm.p2H[c][q] -= g.dt * dc2[c];
    }
    return;
  }
  const ClassEntry ce = mt.table[mt.cls ? mt.cls[q] : 0];
  bool over = false;
  float dv = 0.f;
  if (mt.d_on) {
    const int di = i - mt.d_i0, dj = j - mt.d_j0, dk = k - mt.d_k0;
    if (di >= 0 && di < mt.d_ni && dj >= 0 && dj < mt.d_nj && dk >= 0 && dk < mt.d_nk) {
      dv = mt.d_inv_eps[((long long)di * mt.d_nj + dj) * mt.d_nk + dk];
      over = true;
    }
  }
#pragma unroll
  for (int c = 0; c < 3; c++) {
    if (dc[c] == 0.0f) continue;
    if (!over && (ce.special & (1 << c)) && ade.on) {
      const long long b = (long long)(i - ade.i0) * ade.bsx + (long long)(j - ade.j0) * ade.bsy + (k - ade.k0);
      const AdeMat& am = ade.mats[ce.mat[c]];
      const float dE = am.kE[2] * g.dt * dc[c];
      stx(f.E[c], q, ldx(f.E[c], q, sc.ie[c], sc.xz, c, xq) + dE, sc.se[c], sc.xz, c, xq);
      for (int p = 0; p < am.np; p++) ade.Jp[c][p][b] += am.kJ[p][2] * dE;
    } else {
      const float ie = over ? dv : ce.inv_eps[c];
      stx(f.E[c], q, ldx(f.E[c], q, sc.ie[c], sc.xz, c, xq) + g.dt * ie * dc[c], sc.se[c], sc.xz, c, xq);
      if (dc2[c] != 0.0f) pm.p2E[c][q] += g.dt * ie * dc2[c];
    }
  }
}

constexpr int kOff[6][3] = {{0, 1, 1}, {1, 0, 1}, {1, 1, 0}, {1, 0, 0}, {0, 1, 0}, {0, 0, 1}};

// Incident field evaluated at every point.  Bound by its FP64 instructions
// (sines and exponentials) at three waves a SIMD; the axis is a scalar and no
// array is indexed by it, or the grid's constants go to scratch memory and
// registers for two waves are left.  Both launches of a step, oblique wave: 128^3
// 68.0 us so, 49.6 now; 256^3 215 and 139; dipole box of 40^3 cells 69.7 and 63.5.
// (One copy of the evaluation for the four neighbours too: 50.8, 143, 66.6.)
template <int STORE, int MODE>
__global__ __launch_bounds__(256) void k_tfsf(Grid g, Fields<STORE> f, Scales sc, Cpml pm, Materials mt, Ade ade,
                                              Tfsf tf, TfsfBands bands, double tinc) {
  int r, i, j, k;
  if (!band_cell(bands, r, i, j, k)) return;
  r = __builtin_amdgcn_readfirstlane(r);
  float dc[3] = {0.f, 0.f, 0.f}, dc2[3] = {0.f, 0.f, 0.f};
#pragma nounroll
  for (int rb = r; rb < bands.n; rb++) {
    if (rb != r && !band_has(bands, r, rb, i, j, k)) continue;
    const int a = __builtin_amdgcn_readfirstlane(bands.axis[rb]), b1 = a == 2 ? 0 : a + 1, b2 = a == 0 ? 2 : a - 1;
    // components with a derivative along a: b2 (first curl term), b1 (second)
#pragma nounroll
    for (int t = 0; t < 2; t++) {
      const int c = t == 0 ? b2 : b1, cq = (MODE == 1 ? 3 : 0) + (t == 0 ? b1 : b2);
      auto half = [&](int v, int e) { return 2 * v + ((e == c) == (MODE == 1) ? 0 : 1); };
      const float rd0 = g.rd[0], rd1 = g.rd[1], rd2 = g.rd[2], rd = a == 0 ? rd0 : (a == 1 ? rd1 : rd2);
      const float D = rd * tfsf_dcorr(tf, half(i, 0), half(j, 1), half(k, 2), a, cq, tinc);
      if (D == 0.0f) continue;
      tfsf_term<MODE>(g, pm, a, c, t, D, i, j, k, dc, dc2);
    }
  }
  tfsf_apply<STORE, MODE>(g, f, sc, pm, mt, ade, i, j, k, dc, dc2);
}

// One point of a dipole's table (Tfsf::ptab) at time t.
__device__ __forceinline__ void tfsf_point(const Tfsf& tf, double* out, long long q, double t) {
  const long long n = 6LL * tf.ptab_n[0] * tf.ptab_n[1] * tf.ptab_n[2];
  if (q >= n) return;  // n < 2^31 (kMaxPointTable)
  const unsigned n1 = tf.ptab_n[1], n2 = tf.ptab_n[2], u = (unsigned)q;
  const int p2 = (int)(u % n2);
  const unsigned r = u / n2;
  const int p1 = (int)(r % n1);
  const int p0 = (int)((r / n1) % (unsigned)tf.ptab_n[0]);
  const int c = (int)(r / n1 / (unsigned)tf.ptab_n[0]);
  out[q] = incident(tf, c, tf.ptab_h0[0] + p0, tf.ptab_h0[1] + p1, tf.ptab_h0[2] + p2, t);
}

// Incident field from a table: TAB 1 of a plane wave along an axis, per
// half-coordinate; TAB 2 of a small dipole box, per point.  The axes and
// components are unrolled: which component a stencil reads, and all its
// indices, are then known, and the table values of a cell are loaded together.
// A dipole's launch takes every cell around its box (bands.r[0]) instead of
// the face bands, and its blocks from nblk on fill the table of the next
// half-step.  Bound by its chain of loads: the table, the cell's fields, the
// store.  A dipole box of 4^3 cells: 5.8 us (H) and 6.7 us (E), against 18.4,
// 18.8 and 4.6 for each table's own launch with axis, component and neighbour
// in nested loops.  Plane wave along z, 128x128 cells on two faces: 5.8 and
// 6.8 us against 7.1 and 7.7.
template <int STORE, int MODE, int TAB>
__global__ __launch_bounds__(256) void k_tfsf_tab(Grid g, Fields<STORE> f, Scales sc, Cpml pm, Materials mt, Ade ade,
                                                  Tfsf tf, TfsfBands bands, unsigned nblk) {
  if (TAB == 2 && blockIdx.x >= nblk) {
    tfsf_point(tf, tf.pnext, (blockIdx.x - nblk) * 256LL + threadIdx.x, tf.tnext);
    return;
  }
  int i, j, k;
  if constexpr (TAB == 2) {
    const Region& R = bands.r[0];
    const unsigned nk = (unsigned)(R.k1 - R.k0), nj = (unsigned)(R.j1 - R.j0);
    const unsigned loc = blockIdx.x * 256 + threadIdx.x, row = loc / nk;
    if (loc >= nk * nj * (unsigned)(R.i1 - R.i0)) return;
    k = R.k0 + (int)(loc - row * nk);
    j = R.j0 + (int)(row % nj);
    i = R.i0 + (int)(row / nj);
  } else {
    int r;
    if (!band_cell(bands, r, i, j, k)) return;
  }
  const int v[3] = {i, j, k};
  const int ho[4] = {-3, -1, 1, 3};
  const double wt[4] = {1.0, -27.0, 27.0, -1.0};
  float dc[3] = {0.f, 0.f, 0.f}, dc2[3] = {0.f, 0.f, 0.f}, D[3][2];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    const int b1 = (a + 1) % 3, b2 = (a + 2) % 3;
    const bool face = (v[a] >= tf.fl0[a] && v[a] <= tf.fl1[a]) || (v[a] >= tf.fh0[a] && v[a] <= tf.fh1[a]);
    D[a][0] = D[a][1] = 0.f;
    // (a wave of one band has two axes without a face)
    if (TAB == 1 && __builtin_amdgcn_ballot_w64(face) == 0) continue;
#pragma unroll
    for (int t = 0; t < 2; t++) {
      const int c = t == 0 ? b2 : b1;
      const int comp = MODE == 1 ? c : 3 + c;                       // updated
      const int cq = (MODE == 1 ? 3 : 0) + (t == 0 ? b1 : b2);      // read across the face
      const int h[3] = {2 * i + kOff[comp][0], 2 * j + kOff[comp][1], 2 * k + kOff[comp][2]};
      const bool in = h[b1] >= tf.hlo[b1] && h[b1] <= tf.hhi[b1] && h[b2] >= tf.hlo[b2] && h[b2] <= tf.hhi[b2];
      const bool pin = h[a] >= tf.hlo[a] && h[a] <= tf.hhi[a];
      double acc = 0.0;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int hq = h[a] + ho[q];
        const bool qin = hq >= tf.hlo[a] && hq <= tf.hhi[a];
        const bool need = in && qin != pin;
        double x;
        if constexpr (TAB == 1) {
          const int ha = tf.tab_axis == a ? hq : h[tf.tab_axis == b1 ? b1 : b2];
          x = tf.P[cq] * tf.table[min(max(ha - tf.tab_h0, 0), tf.tab_n - 1)];
        } else {
          int p[3];
#pragma unroll
          for (int e = 0; e < 3; e++) p[e] = (e == a ? hq : h[e]) - tf.ptab_h0[e];
          const int at = ((cq * tf.ptab_n[0] + p[0]) * tf.ptab_n[1] + p[1]) * tf.ptab_n[2] + p[2];
          x = tf.ptab[need ? at : 0];  // a needed point lies in the table
        }
        const bool qsf = tf.sf_inside ? qin : !qin;  // the neighbour is in the scattered-field region
        acc += wt[q] * (need ? (qsf ? x : -x) : 0.0);
      }
      D[a][t] = g.rd[a] * (float)acc;
    }
  }
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int t = 0; t < 2; t++)
      if (D[a][t] != 0.0f)
        tfsf_term<MODE>(g, pm, a, t == 0 ? (a + 2) % 3 : (a + 1) % 3, t, D[a][t], i, j, k, dc, dc2);
  tfsf_apply<STORE, MODE>(g, f, sc, pm, mt, ade, i, j, k, dc, dc2);
}

// Plane-wave waveform along the propagation axis, one value per
// half-coordinate: with k parallel to axis a the incident phase depends on
// the half-coordinate along a only (signal.hpp:17-26).  One launch fills the
// tables of nsteps steps, both half-steps: out[(s*2 + half)*tab_n + h] at
// t = (n0+s) dt (H half, incident E) and (n0+s+1/2) dt (E half, incident H).
__global__ __launch_bounds__(256) void k_tfsf_table(Tfsf tf, double* out, long long n0, int nsteps, double dt) {
  const long long idx = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (idx >= (long long)nsteps * 2 * tf.tab_n) return;
  const int h = (int)(idx % tf.tab_n);
  const int half = (int)((idx / tf.tab_n) % 2);
  const long long n = n0 + idx / (2LL * tf.tab_n);
  const double t = half ? ((double)n + 0.5) * dt : (double)n * dt;
  const int a = tf.tab_axis;
  const double ka = a == 0 ? tf.kx : (a == 1 ? tf.ky : tf.kz);
  const double xa = (h + tf.tab_h0) * tf.half_d[a];
  double f0, f1, f2;
  wave3(tf.waveform, tf.w * t - ka * (xa - tf.pos[a]), tf.w, tf.kEnv, tf.t0, tf.tw, f0, f1, f2);
  out[idx] = tf.amp * f0;
}

// ======================================================== small kernels
template <int STORE>
__global__ void k_soft(Fields<STORE> f, Scales sc, Soft so) {
  const int t = threadIdx.x;
  if (t >= so.n) return;
  const int c = so.comp[t];
  const long long q = so.q[t];
  const int xq = STORE == 1 ? exact_idx(sc.xz, so.ijk[t][0], so.ijk[t][1], so.ijk[t][2]) : -1;
  stx(f.E[c], q, ldx(f.E[c], q, sc.ie[c], sc.xz, c, xq) - so.val[t], sc.se[c], sc.xz, c, xq);
}

template <int STORE>
__global__ void k_record(Grid g, Fields<STORE> f, Scales sc, Probes pr, int fields) {
  record_thread(pr, blockIdx.x * (long long)blockDim.x + threadIdx.x, fields, [&](int comp, int i, int j, int k) {
    const int ii = nbr(i, 0, g.nx, g.per[0]), jj = nbr(j, 0, g.ny, g.per[1]), kk = nbr(k, 0, g.nz, g.per[2]);
    if (ii < 0 || jj < 0 || kk < 0) return 0.f;
    const long long q = ii * g.sx + jj * g.sy + kk;
    const int xq = STORE == 1 ? exact_idx(sc.xz, ii, jj, kk) : -1;
    return comp < 3 ? ldx(f.E[comp], q, sc.ie[comp], sc.xz, comp, xq)
                    : ldx(f.H[comp - 3], q, sc.ih[comp - 3], sc.xz, comp, xq);
  });
}

__global__ void k_to_float_h(const __half* src, float inv, float* dst, long long n) {
  for (long long q = blockIdx.x * (long long)blockDim.x + threadIdx.x; q < n; q += (long long)gridDim.x * blockDim.x)
    dst[q] = __half2float(src[q]) * inv;
}
__global__ void k_from_float_h(const float* src, float s, __half* dst, long long n) {
  for (long long q = blockIdx.x * (long long)blockDim.x + threadIdx.x; q < n; q += (long long)gridDim.x * blockDim.x)
    dst[q] = __float2half_rn(src[q] * s);
}

// ============================================================ launchers
// First failed or refused launch of this thread since the last
// take_launch_error (kernel name and reason).
static thread_local char t_launch_err[256];
static thread_local bool t_launch_failed = false;

void fail_launch(const char* kernel, const char* why) {
  if (t_launch_failed) return;  // keep the first
  snprintf(t_launch_err, sizeof(t_launch_err), "launch of %s failed: %s", kernel, why);
  t_launch_failed = true;
}

void note_launch(const char* kernel) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) fail_launch(kernel, hipGetErrorString(e));
}

int take_launch_error(char* msg, int cap) {
  if (!t_launch_failed) return 0;
  if (msg && cap > 0) snprintf(msg, (size_t)cap, "%s", t_launch_err);
  t_launch_failed = false;
  return 1;
}

static void check_launch(const char* what) { note_launch(what); }

// One launch over the union of the face bands (k_tfsf gives each cell one
// writer); the host fills each band's first thread index and its overlap
// mask.
static unsigned point_blocks(const Tfsf& tf) {
  return (unsigned)((6LL * tf.ptab_n[0] * tf.ptab_n[1] * tf.ptab_n[2] + 255) / 256);
}
template <int STORE, int MODE>
static void tfsf_go(const Grid& g, const void* fields, const Scales& sc, const Cpml& pm, const Materials& mt,
                    const Ade& ade, const Tfsf& tf, const TfsfBands& bands, double tinc, hipStream_t st) {
  const Fields<STORE>& f = *static_cast<const Fields<STORE>*>(fields);
  if (tf.ptab) {  // a dipole with a table: the cells around its box
    TfsfBands b{};
    const int dim[3] = {g.nx, g.ny, g.nz};
    int lo[3], hi[3];
    long long n = 1;
    for (int a = 0; a < 3; a++) {
      lo[a] = std::max(tf.fl0[a], 0);
      hi[a] = std::min(tf.fh1[a] + 1, dim[a]);
      n *= std::max(hi[a] - lo[a], 0);
    }
    if (n == 0 || bands.n == 0) return;
    b.n = 1;
    b.r[0] = Region{lo[0], hi[0], lo[1], hi[1], lo[2], hi[2]};
    const unsigned nblk = (unsigned)((n + 255) / 256);
    const unsigned more = tf.pnext ? point_blocks(tf) : 0;
    hipLaunchKernelGGL((k_tfsf_tab<STORE, MODE, 2>), dim3(nblk + more), dim3(256), 0, st, g, f, sc, pm, mt, ade, tf,
                       b, nblk);
    check_launch("k_tfsf_tab");
    return;
  }
  TfsfBands b = bands;
  long long n = 0;
  b.start[0] = 0;
  for (int r = 0; r < b.n; r++) {
    const Region& R = b.r[r];
    n += ((long long)(R.i1 - R.i0) * (R.j1 - R.j0) * (R.k1 - R.k0) + 63) / 64 * 64;  // wavefront-aligned
    b.start[r + 1] = (unsigned)std::min<long long>(n, 0xffffffffLL);
    b.ovl[r] = 0;
    for (int q = 0; q < b.n; q++) {
      const Region& Q = b.r[q];
      if (q != r && R.i0 < Q.i1 && Q.i0 < R.i1 && R.j0 < Q.j1 && Q.j0 < R.j1 && R.k0 < Q.k1 && Q.k0 < R.k1)
        b.ovl[r] |= 1u << q;
    }
  }
  if (n <= 0) return;
  if (n >= (1LL << 31)) {  // dtm_create rejects such boxes; never index past 2^31 threads
    fail_launch("k_tfsf", "TF/SF face bands hold 2^31 cells or more");
    return;
  }
  const unsigned nblk = (unsigned)((n + 255) / 256);
  if (tf.tab_axis >= 0)
    hipLaunchKernelGGL((k_tfsf_tab<STORE, MODE, 1>), dim3(nblk), dim3(256), 0, st, g, f, sc, pm, mt, ade, tf, b, nblk);
  else
    hipLaunchKernelGGL((k_tfsf<STORE, MODE>), dim3(nblk), dim3(256), 0, st, g, f, sc, pm, mt, ade, tf, b, tinc);
  check_launch("k_tfsf");
}

void launch_tfsf_tables(const Tfsf& tf, double* out, long long n0, int nsteps, double dt, hipStream_t st) {
  const long long n = (long long)nsteps * 2 * tf.tab_n;
  hipLaunchKernelGGL(k_tfsf_table, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, tf, out, n0, nsteps, dt);
  check_launch("k_tfsf_table");
}

// Per-plane factors of the folded TF/SF source (plane wave along x) for the
// half-steps of a table batch: out[(s*2 + half)*(nx+1)*kFoldStride] holds the
// header, then plane i's six factors at +kFoldStride*(1+i).  tables: the
// batch's waveform tables (k_tfsf_table).  With T(h) = P-less table value at
// x half-coordinate h, xin(h) = h inside the box on x and
// X(h) = sum over the neighbours h+o across an x face of wt_o (+-1) T(h+o):
//   H half: rd1 xin(2i+1) P[Ez] T(2i+1), rd2 xin(2i+1) P[Ey] T(2i+1),
//           rd2 xin(2i) P[Ex] T(2i),     rd0 P[Ez] X(2i), rd0 P[Ey] X(2i),
//           rd1 xin(2i) P[Ex] T(2i);
//   E half: rd1 xin(2i) P[Hz] T(2i),     rd2 xin(2i) P[Hy] T(2i),
//           rd2 xin(2i+1) P[Hx] T(2i+1), rd0 P[Hz] X(2i+1), rd0 P[Hy] X(2i+1),
//           rd1 xin(2i+1) P[Hx] T(2i+1).
__global__ __launch_bounds__(256) void k_tfsf_fold(Tfsf tf, const double* tables, float* out, int nsteps, int nx,
                                                   float rd0, float rd1, float rd2) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  const int per = nx + 1;
  if (idx >= nsteps * 2 * per) return;
  const int sh = idx / per, p = idx % per;  // sh = step * 2 + half
  const int half = sh & 1;
  float* o = out + (long long)sh * per * kFoldStride;
  if (p == 0) {  // header
    int* hd = reinterpret_cast<int*>(o);
    hd[0] = tf.hlo[1];
    hd[1] = tf.hhi[1];
    hd[2] = tf.hlo[2];
    hd[3] = tf.hhi[2];
    hd[4] = tf.sf_inside;
    hd[5] = hd[6] = hd[7] = 0;
    return;
  }
  const int i = p - 1;
  const double* T = tables + (long long)sh * tf.tab_n;
  auto Tv = [&](int h) { return T[min(max(h - tf.tab_h0, 0), tf.tab_n - 1)]; };
  auto xin = [&](int h) { return h >= tf.hlo[0] && h <= tf.hhi[0] ? 1.0 : 0.0; };
  auto X = [&](int h) {
    const bool pin = h >= tf.hlo[0] && h <= tf.hhi[0];
    const int ho[4] = {-3, -1, 1, 3};
    const double wt[4] = {1.0, -27.0, 27.0, -1.0};
    double acc = 0.0;
    for (int q = 0; q < 4; q++) {
      const int hq = h + ho[q];
      const bool qin = hq >= tf.hlo[0] && hq <= tf.hhi[0];
      if (qin == pin) continue;
      const double v = Tv(hq);
      acc += wt[q] * ((tf.sf_inside ? qin : !qin) ? v : -v);
    }
    return acc;
  };
  const int e = 2 * i, od = 2 * i + 1;
  float* u = o + kFoldStride * p;
  if (half == 0) {  // neighbours are E components (0, 1, 2)
    u[0] = (float)(rd1 * xin(od) * tf.P[2] * Tv(od));
    u[1] = (float)(rd2 * xin(od) * tf.P[1] * Tv(od));
    u[2] = (float)(rd2 * xin(e) * tf.P[0] * Tv(e));
    u[3] = (float)(rd0 * tf.P[2] * X(e));
    u[4] = (float)(rd0 * tf.P[1] * X(e));
    u[5] = (float)(rd1 * xin(e) * tf.P[0] * Tv(e));
  } else {          // neighbours are H components (3, 4, 5)
    u[0] = (float)(rd1 * xin(e) * tf.P[5] * Tv(e));
    u[1] = (float)(rd2 * xin(e) * tf.P[4] * Tv(e));
    u[2] = (float)(rd2 * xin(od) * tf.P[3] * Tv(od));
    u[3] = (float)(rd0 * tf.P[5] * X(od));
    u[4] = (float)(rd0 * tf.P[4] * X(od));
    u[5] = (float)(rd1 * xin(od) * tf.P[3] * Tv(od));
  }
  u[6] = u[7] = 0.f;
}

void launch_tfsf_fold(const Tfsf& tf, const double* tables, float* out, int nsteps, const Grid& g,
                      hipStream_t st) {
  const int n = nsteps * 2 * (g.nx + 1);
  hipLaunchKernelGGL(k_tfsf_fold, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, tf, tables, out, nsteps,
                     g.nx, g.rd[0], g.rd[1], g.rd[2]);
  check_launch("k_tfsf_fold");
}

// Incident values of every component on the point table's box at time t:
// one thread per value, so the FP64 transcendentals of a dipole run across
// the chip instead of in the band threads one after another.
__global__ __launch_bounds__(256) void k_tfsf_points(Tfsf tf, double t) {
  tfsf_point(tf, tf.ptab, blockIdx.x * 256LL + threadIdx.x, t);
}

void launch_tfsf(int store, int half, const Grid& g, const void* fields, const Scales& sc, const Cpml& pm,
                 const Materials& mt, const Ade& ade, const Tfsf& tf, const TfsfBands& bands, double t_inc,
                 hipStream_t st) {
  if (tf.ptab && !tf.pfull) {
    hipLaunchKernelGGL(k_tfsf_points, dim3(point_blocks(tf)), dim3(256), 0, st, tf, t_inc);
    check_launch("k_tfsf_points");
  }
  if (store == 0 && half == 0) tfsf_go<0, 0>(g, fields, sc, pm, mt, ade, tf, bands, t_inc, st);
  if (store == 0 && half == 1) tfsf_go<0, 1>(g, fields, sc, pm, mt, ade, tf, bands, t_inc, st);
  if (store == 0 && half == 2) tfsf_go<0, 2>(g, fields, sc, pm, mt, ade, tf, bands, t_inc, st);
  if (store == 1 && half == 0) tfsf_go<1, 0>(g, fields, sc, pm, mt, ade, tf, bands, t_inc, st);
  if (store == 1 && half == 1) tfsf_go<1, 1>(g, fields, sc, pm, mt, ade, tf, bands, t_inc, st);
  if (store == 1 && half == 2) tfsf_go<1, 2>(g, fields, sc, pm, mt, ade, tf, bands, t_inc, st);
}

// The variant with room for the poles of the box (0: conductive or gyrotropic cells only).
template <int STORE, bool XZ>
static void ade_go(const Grid& g, const Fields<STORE>& f, const Fields<STORE>& fd, const Scales& sc,
                   const Materials& mt, const Ade& ade, hipStream_t st) {
  AdeArgs<STORE> A{};
  A.ni = ade.ni;
  A.nj = ade.nj;
  A.nk = ade.nk;
  A.i0 = ade.i0;
  A.j0 = ade.j0;
  A.k0 = ade.k0;
  A.sx = g.sx;
  A.sy = g.sy;
  A.dt = g.dt;
  A.cls = mt.cls;
  A.table = mt.table;
  A.mats = ade.mats;
  A.gmats = ade.gmats;
  A.wide = mt.nclass > 32;
  for (int w = 0; w < kMaxClasses / 32; w++) A.special[w] = ade.special[w];
  A.d_on = mt.d_on;
  const int d0[3] = {mt.d_i0, mt.d_j0, mt.d_k0}, dn[3] = {mt.d_ni, mt.d_nj, mt.d_nk};
  for (int c = 0; c < 3; c++) {
    A.E[c] = f.E[c];
    A.Ed[c] = fd.E[c];
    A.ie[c] = sc.ie[c];
    A.se[c] = sc.se[c];
    A.curl[c] = ade.curl[c];
    A.Em[c] = ade.Em[c];
    A.Jg[c] = ade.Jg[c];
    for (int p = 0; p < kMaxPoles; p++) {
      // (the variant may read, but never use, a pole more than the box has arrays for)
      A.Jp[c][p] = p < ade.npoles ? ade.Jp[c][p] : ade.Em[c];
      A.Jm[c][p] = p < ade.npoles ? ade.Jm[c][p] : ade.Em[c];
    }
    A.d0[c] = d0[c];
    A.dn[c] = dn[c];
  }
  A.xz = sc.xz;
  box_launches((unsigned)ade.ni, (unsigned long long)ade.nj * ade.nk, [&](const BoxUnits& un, unsigned blocks) {
    A.un = un;
    auto run = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kBoxBlock), 0, st, A); };
    if (ade.gyro_on) {
      if (ade.npoles > 2) run(k_ade<STORE, 4, true, XZ>);
      else if (ade.npoles > 0) run(k_ade<STORE, 2, true, XZ>);
      else run(k_ade<STORE, 0, true, XZ>);
    } else {
      if (ade.npoles > 2) run(k_ade<STORE, 4, false, XZ>);
      else if (ade.npoles > 1) run(k_ade<STORE, 2, false, XZ>);
      else if (ade.npoles > 0) run(k_ade<STORE, 1, false, XZ>);
      else run(k_ade<STORE, 0, false, XZ>);
    }
  });
  check_launch("k_ade");
}

void launch_ade(int store, const Grid& g, const void* fsrc, const void* fdst, const Scales& sc, const Materials& mt,
                const Ade& ade, hipStream_t st) {
  if (!ade.on) return;
  if (store == 0)
    ade_go<0, false>(g, *static_cast<const Fields<0>*>(fsrc), *static_cast<const Fields<0>*>(fdst), sc, mt, ade, st);
  else if (sc.xz.on)
    ade_go<1, true>(g, *static_cast<const Fields<1>*>(fsrc), *static_cast<const Fields<1>*>(fdst), sc, mt, ade, st);
  else
    ade_go<1, false>(g, *static_cast<const Fields<1>*>(fsrc), *static_cast<const Fields<1>*>(fdst), sc, mt, ade, st);
}

void launch_soft(int store, const Grid&, const void* fields, const Scales& sc, const Soft& so, hipStream_t st) {
  if (so.n <= 0) return;
  if (store == 0)
    hipLaunchKernelGGL(k_soft<0>, dim3(1), dim3(64), 0, st, *static_cast<const Fields<0>*>(fields), sc, so);
  else
    hipLaunchKernelGGL(k_soft<1>, dim3(1), dim3(64), 0, st, *static_cast<const Fields<1>*>(fields), sc, so);
  check_launch("k_soft");
}

void launch_record(int store, const Grid& g, const void* fields, const Scales& sc, const Probes& pr, int which,
                   hipStream_t st) {
  if (pr.n <= 0) return;
  const unsigned nb = (unsigned)((record_threads(pr) + 63) / 64);
  if (store == 0)
    hipLaunchKernelGGL(k_record<0>, dim3(nb), dim3(64), 0, st, g, *static_cast<const Fields<0>*>(fields), sc, pr, which);
  else
    hipLaunchKernelGGL(k_record<1>, dim3(nb), dim3(64), 0, st, g, *static_cast<const Fields<1>*>(fields), sc, pr, which);
  check_launch("k_record");
}

void launch_to_float(int store, const void* src, float inv, float* dst, long long n, hipStream_t st) {
  if (store == 0) {
    if (hipMemcpyAsync(dst, src, sizeof(float) * n, hipMemcpyDeviceToDevice, st) != hipSuccess)
      fail_launch("field copy", hipGetErrorString(hipGetLastError()));
    return;
  }
  hipLaunchKernelGGL(k_to_float_h, dim3(1024), dim3(256), 0, st, static_cast<const __half*>(src), inv, dst, n);
  check_launch("k_to_float_h");
}

void launch_from_float(int store, const float* src, float s, void* dst, long long n, hipStream_t st) {
  if (store == 0) {
    if (hipMemcpyAsync(dst, src, sizeof(float) * n, hipMemcpyDeviceToDevice, st) != hipSuccess)
      fail_launch("field copy", hipGetErrorString(hipGetLastError()));
    return;
  }
  hipLaunchKernelGGL(k_from_float_h, dim3(1024), dim3(256), 0, st, src, s, static_cast<__half*>(dst), n);
  check_launch("k_from_float_h");
}

const char* kernel_variant_name(int store) {
  return store == 0 ? "k_sweep<fp32>" : "k_sweep<fp16>";
}

}  // namespace dtm
