// dtm_probe.h — recording of probes and sensors, by a launch of its own
// (k_record) or by blocks of the sweeps' launches.
#pragma once
#include "dtm_internal.h"

namespace dtm {

// get(comp, i, j, k): field value with the boundary rule.
// Reference sensor interpolation (sensor.h:64-71) on the cell lattice.
template <typename Get> __device__ __forceinline__ float sensor_val(Get get, int comp, int x, int y, int z) {
  const int zM = (z == 0) ? z + 1 : z - 1;
  switch (comp) {
    case 0: return 0.25f * (get(0, x, y - 1, zM) + get(0, x, y - 1, z) + get(0, x, y, zM) + get(0, x, y, z));
    case 1: return 0.25f * (get(1, x - 1, y, zM) + get(1, x - 1, y, z) + get(1, x, y, zM) + get(1, x, y, z));
    case 2: return 0.25f * (get(2, x - 1, y - 1, z) + get(2, x - 1, y, z) + get(2, x, y - 1, z) + get(2, x, y, z));
    case 3: return 0.5f * (get(3, x - 1, y, z) + get(3, x, y, z));
    case 4: return 0.5f * (get(4, x, y - 1, z) + get(4, x, y, z));
    default: return 0.5f * (get(5, x, y, zM) + get(5, x, y, z));
  }
}

// One thread per (probe, DFT bin): every thread of a probe reads its value
// (a few cached loads), the bin-0 thread stores it to the series, and each
// thread advances its own FP64 accumulator, so the sincos of the bins run in
// parallel rather than one after another (64 bins: 26 -> 5 us per step).
// fields: bit 0: probes of E components, bit 1: of H components.
template <typename Get>
__device__ __forceinline__ void record_thread(const Probes& pr, long long tid, int fields, Get get) {
  const int nb = pr.nfreq > 0 ? pr.nfreq : 1;
  if (tid >= (long long)pr.n * nb) return;
  int p, fq;
  if (tid >> 31) {
    p = (int)(tid / nb);
    fq = (int)(tid % nb);
  } else {
    p = (int)((unsigned)tid / (unsigned)nb);
    fq = (int)((unsigned)tid % (unsigned)nb);
  }
  const ProbeDesc d = pr.desc[p];
  if (!(fields & (d.comp < 3 ? 1 : 2)) || d.i < pr.i0 || d.i >= pr.i1) return;
  const float v = d.kind == 0 ? get(d.comp, d.i, d.j, d.k) : sensor_val(get, d.comp, d.i, d.j, d.k);
  if (fq == 0) pr.series[(long long)pr.row * pr.n + p] = v;
  if (pr.nfreq > 0) {
    const double t = d.comp < 3 ? (double)(pr.step + 1) * pr.dt : ((double)pr.step + 0.5) * pr.dt;
    double* acc = pr.dft + ((long long)p * pr.nfreq + fq) * 2;
    double s, c;
    sincos(pr.omega[fq] * t, &s, &c);
    acc[0] += (double)v * c * pr.dt;
    acc[1] += (double)v * s * pr.dt;
  }
}
inline long long record_threads(const Probes& pr) { return (long long)pr.n * (pr.nfreq > 0 ? pr.nfreq : 1); }

}  // namespace dtm
