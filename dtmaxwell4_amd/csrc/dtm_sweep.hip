// dtm_sweep.hip — the H and E half-step sweeps.
//
//   H^{n+1/2} = H^{n-1/2} - dt curl E^n          (genAlg.py:182-301, time 0)
//   E^{n+1}   = E^n + dt/eps curl H^{n+1/2}      (time 1/2)
// with the (2,4) difference D f = [27 (f_{+1/2} - f_{-1/2}) - (f_{+3/2} - f_{-3/2})]/(24 d)
// (defs.h:3-13) on the cell lattice of include/dtmaxwell4.h.
//
// One kernel for both half-steps (UP 0: H from E, UP 1: E from H): the two
// differ by the direction in which their stencils reach, i-2 .. i+1 against
// i-1 .. i+2 along every axis, and by the material factor.
//
// A lane owns a chunk of four consecutive z cells of one (x, y) row: one
// 16-byte load (8 bytes in half storage) per component, and a quarter of the
// index arithmetic, branches and scalar work per cell.  The rows of an x plane
// are laid end to end, so lane L of a plane holds chunk L % nzv of row L / nzv
// and no lane idles for a z extent that is no multiple of a tile.  A lane
// marches along x over a segment of planes:
//  - the x stencil reads a queue of four planes in registers;
//  - the y stencil loads the three other rows, which L1 and the XCD's L2 hold;
//  - the z stencil takes its neighbours from the adjacent lanes (DPP).
// Waves share nothing and never wait for each other: no barrier, and LDS only
// for a lane's own coefficients.
//
// All accesses are buffer loads and stores on one plane: the plane's base is a
// scalar, a lane's offset in the plane does not change along the march, and a
// position outside the grid is an offset beyond the descriptor's range, which
// reads zero and stores nothing.  So no boundary costs a branch, and the index
// arithmetic is a few scalar instructions per plane.
//
// Bounds and figures (us a step of both sweeps, plane wave on a sphere, CPML;
// in brackets the sweeps before these: 64 x 8 or 16 column tiles in LDS with a
// barrier per plane, one cell per lane):
//   512x256x256 FP32  557 (587)  HBM: 88 B/cell (Yee words 73, psi 7.5) at 5.1-5.4 TB/s, a copy 4.7-5.3
//               FP16  348 (471)  HBM and issue: 48 B/cell (Yee words 37, psi 7.5) at 4.5-4.7 TB/s
//   256^3       FP32  302 (316)  FP16 192 (250)
//   200^3       FP32  122 (160)  FP16  82 (148)  fields partly, or all, in the Infinity Cache
//   128^3       FP32   37  (54)  FP16  30  (49)  one or two rounds of waves: latency and issue
//    64^3       FP32   12  (29)  FP16  12  (31)  two launches of one plane per wave: latency
// (whole grid; several steps of a large grid run slab by slab, see skewed_steps).
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "dtm_internal.h"
#include "dtm_probe.h"

namespace dtm {

namespace {

constexpr int NXCD = 8;
constexpr int NV = 4;           // cells of a chunk
constexpr unsigned kFront = 4;  // floats before a psi array that may be read (sdalloc)

using u4 = unsigned __attribute__((ext_vector_type(4)));
using u2 = unsigned __attribute__((ext_vector_type(2)));
using rsrc = __amdgpu_buffer_rsrc_t;

// One launch: blocks [lb0, lb1) of 64 chunks of the planes [i0, i1), without
// blocks [hb0, hb1) of the planes [h0, h1) (the hole, whose planes are below
// h0 = i1 if there is none).  The planes before, of and after the hole are cut
// into segments of seg planes: total[] are the blocks up to the end of each.
// Planes of more than SweepArgs::strip blocks are run strip by strip: all segments
// of the first `strip` blocks of a plane, then those of the next.
struct Sweep {
  int i0, i1, seg, lb0, lb1;
  int h0, h1, hb0, hb1;
  int nzv;             // chunks of a row
  long long NL;        // and of a plane
  int rag;             // nz mod NV: the last chunk of a row is partly outside
  int per, total[3];    // blocks per XCD, and in all
  int zgap;             // cells between the two z slabs
};
// Soft sources that the E sweep subtracts from its new values.
struct SweepSoft {
  int lo, hi;  // their x planes lie in [lo, hi)
  int n;
  int i[kSweepSoft], q[kSweepSoft], comp[kSweepSoft];  // plane, cell of its chunk, component
  long long cell[kSweepSoft];                            // the chunk's first cell in the plane
  float val[kSweepSoft];
};
// The arguments of one half-step: the scales of the three components the curl
// is taken of (src) and of the three it updates (dst), and of the absorbing
// layer the parts that belong to dst.
struct SweepArgs {
  Sweep sw;
  int nx, ny, nz, per[3];
  long long sx;
  float rd[3][3], dt;  // 1/(24 d_a) times the scale of source component c (a power of two: exact)
  char* set;            // Ex Ey Ez Hx Hy Hz, `comp` bytes apart
  unsigned long long comp;
  float isrc[3], idst[3], sdst[3];
  const float* fold;    // this half-step's factor table, and the packed weights of every chunk
  const int2* foldw;
  int pml, plo[3], phi[3];
  int strip;  // of Sweep
  float* psi[3][2];
  const float* b[3];
  const float* c[3];
  float* p2[3];
  Materials mt;
  struct {
    int on, i0, j0, k0;
    long long bsx, bsy;
    float* curl[3];
  } ade;
  Exact xz;
  SweepSoft soft;
  Probes pr;  // probes of src, recorded by the blocks after the sweep's
};
using ArgsK = __attribute__((address_space(4))) const SweepArgs;
// The kernel's own argument block, behind a pointer the compiler cannot see
// through: what is rarely needed is read again there (scalar loads that hit
// the scalar cache) instead of holding scalar registers all along the march.
__device__ __forceinline__ const ArgsK* again() {
  const ArgsK* p = (const ArgsK*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return p;
}

// Touches every line of a kernel's arguments (BYTES of them) at once: the host
// has just written them, so the first waves of an XCD miss each line, and the
// compiler reads them one after the other where they are needed.  FP16: 14.0 ->
// 12.9 us a step at 64^3, 83.0 -> 80.4 at 200^3; FP32 (more waits on fields):
// 12.1 -> 11.9 at 48x40x40, nothing from 64^3 on.
template <int BYTES> __device__ __forceinline__ void prefetch_args() {
  using WordK = __attribute__((address_space(4))) const unsigned;
  WordK* p = (WordK*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  unsigned any = 0;
#pragma unroll
  for (int i = 0; i < BYTES; i += 64) any |= p[i / 4];
  asm volatile("" : : "s"(any));
}

// How a plane of an array is addressed.
//  kNear  the field set is below 4 GiB: one descriptor per plane, based at the
//         plane of Ex, and the component as the scalar offset;
//  kFar   a descriptor per plane and component;
//  kHuge  a plane of 4 GiB or more: 64-bit offsets and flat loads.
enum { kNear, kFar, kHuge };
template <int AD> using Off = typename std::conditional<AD == kHuge, unsigned long long, unsigned>::type;
// an offset beyond every plane
template <int AD> constexpr Off<AD> kOut = AD == kHuge ? (Off<AD>)(1ull << 62) : (Off<AD>)0xffffff00u;
constexpr unsigned long long kBytes = kOut<kNear>;  // what a descriptor spans at most

template <int AD> struct Plane {
  rsrc r;
  unsigned so;
};
template <> struct Plane<kHuge> {
  char* p;  // null: outside the grid
};
// `bytes` from byte0 of base on; none: outside the grid
template <int AD>
__device__ __forceinline__ Plane<AD> span(const void* base, long long byte0, unsigned long long bytes, unsigned so = 0) {
  char* const q = const_cast<char*>(static_cast<const char*>(base)) + byte0;
  if constexpr (AD == kHuge) return Plane<AD>{bytes ? q : nullptr};
  else return Plane<AD>{__builtin_amdgcn_make_buffer_rsrc(q, 0, (int)(unsigned)bytes, 0x00020000), so};
}
template <typename T, int AD> __device__ __forceinline__ T ldt(Plane<AD> p, Off<AD> o) {
  if constexpr (AD == kHuge) {
    T v{};
    if (p.p && o < kOut<AD>) __builtin_memcpy(&v, p.p + o, sizeof(T));
    return v;
  } else {
    const int i = (int)o, so = (int)p.so;
    if constexpr (sizeof(T) == 16) return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b128(p.r, i, so, 0));
    else if constexpr (sizeof(T) == 8) return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(p.r, i, so, 0));
    else if constexpr (sizeof(T) == 4) return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(p.r, i, so, 0));
    else return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b16(p.r, i, so, 0));
  }
}
template <typename T, int AD> __device__ __forceinline__ void stt(Plane<AD> p, Off<AD> o, T v) {
  if constexpr (AD == kHuge) {
    if (p.p && o < kOut<AD>) __builtin_memcpy(p.p + o, &v, sizeof(T));
  } else {
    const int i = (int)o, so = (int)p.so;
    if constexpr (sizeof(T) == 16) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, v), p.r, i, so, 0);
    else if constexpr (sizeof(T) == 8) __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, v), p.r, i, so, 0);
    else if constexpr (sizeof(T) == 4) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), p.r, i, so, 0);
    else __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, v), p.r, i, so, 0);
  }
}

// What a lane holds of a component: stored words (a half keeps its storage form
// until it enters a difference, where the conversion is part of the
// subtraction), or with the FP32 zone floats.
template <typename S, int N> using Vec = S __attribute__((ext_vector_type(N)));
template <int STORE, bool XZ> using Word = typename std::conditional<STORE == 0 || XZ, float, _Float16>::type;
// a chunk, or one cell, of a component
template <int STORE, bool XZ, int AD>
__device__ __forceinline__ Vec<Word<STORE, XZ>, NV> ldw(Plane<AD> p, Off<AD> o, float inv) {
  if constexpr (STORE == 1 && XZ) {
    const auto h = ldt<Vec<_Float16, NV>>(p, o);
    Vec<float, NV> v;
#pragma unroll
    for (int q = 0; q < NV; q++) v[q] = __builtin_fmaf((float)h[q], inv, 0.0f);
    return v;
  } else {
    return ldt<Vec<Word<STORE, XZ>, NV>>(p, o);
  }
}
template <int STORE, bool XZ, int AD>
__device__ __forceinline__ Word<STORE, XZ> ldw1(Plane<AD> p, Off<AD> o, float inv) {
  if constexpr (STORE == 1 && XZ) return __builtin_fmaf((float)ldt<_Float16>(p, o), inv, 0.0f);
  else return ldt<Word<STORE, XZ>>(p, o);
}
// Difference of two words in FP32.  Halves: a 1 - b with the conversions
// (exact) inside the instruction; `one` is 1.0 from a register the compiler
// cannot see through, or it converts both operands first.
__device__ __forceinline__ float sub(float a, float b, float) { return a - b; }
__device__ __forceinline__ float sub(_Float16 a, _Float16 b, float one) {
  return __builtin_fmaf((float)a, one, -(float)b);
}
// (2,4) difference with weights (+1, -27, +27, -1) (genAlg.py:196-198, sign folded)
template <typename S>
__device__ __forceinline__ float d24(S f0, S f1, S f2, S f3, float one) {
  return __builtin_fmaf(27.0f, sub(f2, f1, one), -sub(f3, f0, one));
}

template <int CTRL>
__device__ __forceinline__ unsigned dpp(unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true);
}
constexpr int kFromLower = 0x138;  // wave_shr:1, lane n reads lane n-1
constexpr int kFromUpper = 0x130;  // wave_shl:1, lane n reads lane n+1

// The cells k-2+UP .. k+NV+UP around a lane's NV along z, as e[0 .. NV+2].
template <int UP, typename S>
__device__ __forceinline__ void around(Vec<S, NV> v, S* e) {
  constexpr int NW = NV * (int)sizeof(S) / 4;  // registers
  using W = unsigned __attribute__((ext_vector_type(NW)));
  const W w = __builtin_bit_cast(W, v);
  if constexpr (sizeof(S) == 4) {
#pragma unroll
    for (int t = 0; t < 2 - UP; t++) e[t] = __builtin_bit_cast(S, dpp<kFromLower>(w[NV - 2 + UP + t]));
#pragma unroll
    for (int t = 0; t < 1 + UP; t++) e[2 - UP + NV + t] = __builtin_bit_cast(S, dpp<kFromUpper>(w[t]));
  } else {
    const auto lo = __builtin_bit_cast(Vec<S, 2>, dpp<kFromLower>(w[NW - 1]));
    const auto hi = __builtin_bit_cast(Vec<S, 2>, dpp<kFromUpper>(w[0]));
#pragma unroll
    for (int t = 0; t < 2 - UP; t++) e[t] = lo[UP + t];
#pragma unroll
    for (int t = 0; t < 1 + UP; t++) e[2 - UP + NV + t] = hi[t];
  }
#pragma unroll
  for (int q = 0; q < NV; q++) e[2 - UP + q] = v[q];
}

__device__ __forceinline__ int nbr(int v, int n, int per) {
  if (v >= 0 && v < n) return v;
  if (!per) return -1;
  return v < 0 ? v + n : v - n;
}
__device__ __forceinline__ int slab_index(int v, int n, int plo, int phi) {
  if (v < plo) return v;
  if (v >= n - phi) return plo + v - (n - phi);
  return -1;
}
// a product that is rounded before it is added to anything (opaque, or it becomes part of an fma)
__device__ __forceinline__ float mulr(float a, float b) {
  float r = a * b;
  asm("" : "+v"(r));
  return r;
}
// psi <- b psi + c D ; D <- D + psi   (CPML, kappa = 1, alpha = 0)
__device__ __forceinline__ float cpml(float old, float b, float c, float D) { return __builtin_fmaf(b, old, c * D); }

}  // namespace

// GEN: z extents whose rows do not fill whole waves, ragged rows and a
// periodic z axis: a lane at the end of a wave or row loads the z neighbours
// that no adjacent lane holds.  Without it the rows of a wave end where its
// lanes do, or after 1, 2, 4 .. 32 lanes, and the cells beyond a row's ends are
// outside the grid.
// SP: split-field absorbing layer (genAlg.py:117-148) instead of the CPML.
// TF: a plane-wave TF/SF source along x may be folded in: the correction of
// genAlg.py:219-221 is added to the derivative it belongs to, from this
// half-step's factor table.
// XZ: half storage with the FP32 zone.
// SO: soft sources are subtracted from the new E.  Only launches with sources
// run it: in the ragged FP32 sweep the block costs 9 spilled registers, 3 without.
//
// Registers decide the waves per SIMD: four in half storage (128 VGPRs; at
// three the 512x256x256 step took 14% longer), three in FP32 (168; at four it
// spills and takes 25% longer).
template <int UP, int STORE, bool GEN, bool SP, bool TF, bool XZ, int AD, bool SO>
__global__ __launch_bounds__(64, XZ || SP || AD == kHuge ? 2 : (STORE == 1 ? 4 : 3)) void k_sweep(SweepArgs A) {
  using S = Word<STORE, XZ>;
  using V = Vec<S, NV>;
  using F = Vec<float, NV>;
  using O = Off<AD>;
  constexpr O OUT = kOut<AD>;
  constexpr O ES = STORE == 0 ? 4 : 2;  // bytes of a cell
  constexpr int OWN = 2 - UP;           // the lane's own sample among the four of a stencil
  constexpr int LEAD = 1 + UP;          // planes and cells that a stencil reaches ahead
  constexpr bool HALF = STORE == 1 && !XZ;     // differences in stored units
  constexpr int CS = UP ? 3 : 0, CD = UP ? 0 : 3;  // first source and destination component (Ex .. Hz)
  prefetch_args<sizeof(SweepArgs)>();
  const int blk = blockIdx.x;
  // Probes of the field that this launch only reads: blocks of their own beside
  // the sweep's (a launch of their own took 3 us of a 48x40x40 step's 18, and
  // 4.6 us where 64 bins are summed).
  // (The zone's variants have none, the plain launch before them does: with the
  // recorder in it the compiler kept the arguments of one in scratch memory and
  // spilled 54 registers, 38 us for 13.)
  if (!XZ && blk >= A.sw.per * NXCD) {
    const ArgsK* C = again();
    record_thread(A.pr, (blk - A.sw.per * NXCD) * 64LL + threadIdx.x, 1 << UP,
                  [&](int comp, int i, int j, int k) -> float {
                    const int ii = nbr(i, A.nx, A.per[0]), jj = nbr(j, A.ny, A.per[1]), kk = nbr(k, A.nz, A.per[2]);
                    if (ii < 0 || jj < 0 || kk < 0) return 0.f;
                    const int xq = STORE == 1 ? exact_idx(A.xz, ii, jj, kk) : -1;
                    if (xq >= 0) return C->xz.f[comp][xq];
                    const char* p = A.set + A.comp * comp + (ii * A.sx + (long long)jj * A.nz + kk) * (STORE ? 2 : 4);
                    if constexpr (STORE == 0) return *reinterpret_cast<const float*>(p);
                    else return (float)*reinterpret_cast<const _Float16*>(p) * A.isrc[UP ? comp - 3 : comp];
                  });
    return;
  }
  int lid = (blk % NXCD) * A.sw.per + blk / NXCD;  // XCD-contiguous
  if (lid >= A.sw.total[2]) return;
  int nlb = A.sw.lb1 - A.sw.lb0, lo = A.sw.i0, hi = A.sw.h0;
  bool hole = false;
  if (lid >= A.sw.total[1]) {
    lid -= A.sw.total[1];
    lo = A.sw.h1;
    hi = A.sw.i1;
  } else if (lid >= A.sw.total[0]) {
    lid -= A.sw.total[0];
    lo = A.sw.h0;
    hi = A.sw.h1;
    nlb -= A.sw.hb1 - A.sw.hb0;
    hole = true;
  }
  int lb = A.sw.lb0;
  if (nlb > A.strip) {
    const int nseg = (hi - lo + A.sw.seg - 1) / A.sw.seg, sp = lid / (nseg * A.strip);
    lid -= sp * nseg * A.strip;
    lb += sp * A.strip;
    nlb = min(A.strip, nlb - sp * A.strip);
  }
  const int bs = lid / nlb;
  lb += lid - bs * nlb;
  if (hole && lb >= A.sw.hb0) lb += A.sw.hb1 - A.sw.hb0;
  using LI = typename std::conditional<AD == kHuge, long long, int>::type;
  const LI L = (LI)lb * 64 + (int)threadIdx.x;
  int p0 = lo + bs * A.sw.seg, p1 = min(p0 + A.sw.seg, hi);
  // (opaque, or what they are made from stays in registers along the march)
  asm volatile("" : "+s"(p0), "+s"(p1));
  const bool act = L < A.sw.NL;
  const int j = (int)(L / A.sw.nzv), kc = (int)(L - (LI)j * A.sw.nzv), k = NV * kc;
  const int nz = A.nz, perz = A.per[2];
  const O cell = (O)j * (O)nz + (O)k;
  const O own = act ? cell * ES : OUT;
  const int nx = A.nx, perx = A.per[0];
  auto plane = [&](int p) -> int { return nbr(p, nx, perx); };
  // plane p of component c (Ex .. Hz); outside the grid: empty.  A lane reads
  // whole chunks: the last one of an array reaches into its pad (kPad).
  auto at = [&](int p, int c) -> Plane<AD> {
    const long long o = (long long)max(p, 0) * A.sx * (long long)ES;
    if constexpr (AD == kNear) return span<AD>(A.set, o, p < 0 ? 0 : kBytes, (unsigned)A.comp * (unsigned)c);
    else return span<AD>(A.set, o + (long long)A.comp * c, p < 0 ? 0 : (unsigned long long)(A.sx + NV) * ES);
  };

  // A wave's first loads (fold weights, layer coefficients, the queues) go out
  // before the rest of its start is worked out, without a branch, in the order
  // of their use: waiting for one after the other took 1.3 of 13.9 us a step at
  // 64^3 and 1.6 of 39 at 128^3.  The first plane's own loads follow only after
  // waits: for the coefficients on their way to LDS, for the fold weights, and in
  // E for class 0's flag, a load after the queues and so for all of them.
  // packed TF/SF weights of the cells (k_fold_weights)
  int fz = 0, fi = 0;
  if constexpr (TF) {
    const u2 w = ldt<u2>(span<AD>(A.foldw, 0, A.fold ? (unsigned long long)A.sw.NL * 8 : 0), act ? (O)L * 8u : OUT);
    fz = (int)w[0];
    fi = (int)w[1];
  }
  // Cells of the chunk in a z slab (bit q).
  const int zl = A.plo[2], zh = A.phi[2], yl = A.plo[1], yh = A.phi[1];
  const int Pz = zl + zh;
  const int zin = min(max(zl - k, 0), NV), zout = min(max(nz - zh - k, 0), NV);
  unsigned zm = (((1u << zin) - 1u) | ~((1u << zout) - 1u)) & ((1u << min(NV, nz - k)) - 1u);
  zm = act ? zm : 0u;
  const bool zwave = __builtin_amdgcn_ballot_w64(zm != 0) != 0;
  // (a chunk that reaches into both slabs over a gap has no place in psi)
  const bool zboth = !SP && A.sw.zgap > 0 && A.sw.zgap < 3;
  const bool zslab = !SP && zwave && !zboth;
  const int yup = j - (A.ny - yh);
  int yslab = j < yl ? j : yup >= 0 ? yl + yup : -1;  // the row's place in the y slabs
  yslab = act ? yslab : -1;
  const int ysl = SP ? -1 : yslab;
  const bool sy = SP && yslab >= 0;
  const bool ywave = __builtin_amdgcn_ballot_w64(yslab >= 0) != 0;
  F zb = {}, zc = {};
  float by = 0.f, cy = 0.f;
  {
    if (SP ? zwave : zslab) {  // (NV floats follow the coefficients: setup_cpml)
      const O o = zm != 0 ? (O)k * 4u : OUT;
      zb = ldt<F>(span<AD>(A.b[2], 0, (unsigned long long)(nz + NV) * 4), o);
      zc = ldt<F>(span<AD>(A.c[2], 0, (unsigned long long)(nz + NV) * 4), o);
    }
    if (ywave) {
      const O o = yslab >= 0 ? (O)j * 4u : OUT;
      by = ldt<float>(span<AD>(A.b[1], 0, (unsigned long long)A.ny * 4), o);
      cy = ldt<float>(span<AD>(A.c[1], 0, (unsigned long long)A.ny * 4), o);
    }
  }
  // queues of the source's y and z components: sample q of plane i is plane i-OWN+q
  V qy[4], qz[4];
#pragma unroll
  for (int q = 0; q < 3; q++) {
    const int p = plane(p0 - OWN + q);
    qy[q] = ldw<STORE, XZ>(at(p, CS + 1), own, A.isrc[1]);
    qz[q] = ldw<STORE, XZ>(at(p, CS + 2), own, A.isrc[2]);
  }
  auto row = [&](int dj) -> O {
    const int jj = nbr(j + dj, A.ny, A.per[1]);
    return (act && jj >= 0) ? ((O)jj * (O)nz + (O)k) * ES : OUT;
  };
  const O r0 = row(UP ? -1 : -2), r1 = row(UP ? 1 : -1), r2 = row(UP ? 2 : 1);
  const int nv = min(NV, nz - k);  // cells of the chunk inside the grid
  // z neighbours that no adjacent lane holds
  const int lane = threadIdx.x;
  const bool zfirst = kc == 0, zlast = kc == A.sw.nzv - 1;
  const bool zlo = lane == 0 || zfirst, zhi = lane == 63 || zlast;
  O ol[2] = {OUT, OUT}, oh[2] = {OUT, OUT};
  if constexpr (GEN) {
    auto zoff = [&](int kk) -> O {
      const int kw = nbr(kk, nz, perz);
      return (act && kw >= 0) ? ((O)j * (O)nz + (O)kw) * ES : OUT;
    };
#pragma unroll
    for (int t = 0; t < OWN; t++) ol[t] = zlo ? zoff(k - OWN + t) : OUT;
    const int ke = zlast ? nz : k + NV;
#pragma unroll
    for (int t = 0; t < 2; t++) oh[t] = zhi ? zoff(ke + t) : OUT;
  }
  // FP32 zone: values of zone cells come from their FP32 copies
  bool xwave = false;  // the rows and columns that the wave reads meet the zone
  if constexpr (XZ) {
    const Exact& xz = A.xz;
    const bool near = act && (A.per[1] || perz ||
                              (j > xz.j0 - 4 && j < xz.j1 + 3 && k > xz.k0 - NV - 3 && k < xz.k1 + 3));
    xwave = xz.on && __builtin_amdgcn_ballot_w64(near) != 0;
  }
  // a chunk's cells in the zone's z range (bit q); where a row's cells from k
  // on are or would be in a copy, from kFront floats before it (sdalloc)
  unsigned xm = 0;
  if constexpr (XZ) {
#pragma unroll
    for (int q = 0; q < NV; q++)
      if (act && k + q >= A.xz.k0 && k + q < A.xz.k1) xm |= 1u << q;
  }
  auto copy = [&](int comp) -> Plane<AD> {
    const Exact& x = A.xz;
    return span<AD>(x.f[comp], -4LL * (int)kFront,
                    ((unsigned long long)(x.i1 - x.i0) * (x.j1 - x.j0) * (x.k1 - x.k0) + 2 * kFront) * 4);
  };
  auto in_copy = [&](int p, int jj, int kk) -> O {
    const Exact& x = A.xz;
    if (p < x.i0 || p >= x.i1 || jj < x.j0 || jj >= x.j1) return OUT;
    const long long o = ((long long)(p - x.i0) * (x.j1 - x.j0) + (jj - x.j0)) * (x.k1 - x.k0) + (kk - x.k0);
    return (O)(o + kFront) * 4u;
  };
  auto zone = [&](V& v, int comp, int p, int dj) {
    if constexpr (XZ) {
      const O o = xm != 0 ? in_copy(p, nbr(j + dj, A.ny, A.per[1]), k) : OUT;
      const F z = ldt<F>(copy(comp), o);
#pragma unroll
      for (int q = 0; q < NV; q++) v[q] = o != OUT && ((xm >> q) & 1u) ? z[q] : v[q];
    }
  };
  auto zone1 = [&](S& v, int comp, int p, int kk) {
    if constexpr (XZ) {
      const int kw = nbr(kk, nz, perz);
      const O o = act && kw >= A.xz.k0 && kw < A.xz.k1 ? in_copy(p, j, kw) : OUT;
      const float z = ldt<float>(copy(comp), o);
      v = o != OUT ? z : v;
    }
  };

  // places in psi: of the row, and of the chunk's first cell, where it is or
  // would be: the cells of a slab are contiguous there
  const O oy = ysl >= 0 ? ((O)ysl * (O)nz + (O)k) * 4u : OUT;
  const O oz = zm != 0 ? (O)((long long)j * Pz + (k < zl ? k : k - A.sw.zgap) + (int)kFront) * 4u : OUT;
  // z coefficients of the layer wait in the lane's own LDS slot (nothing is shared)
  __shared__ F lcoef[SP ? 1 : 2][SP ? 1 : 64];
  if constexpr (!SP) {
    if (zslab && zm != 0) {
      lcoef[0][lane] = zb;
      lcoef[SP ? 0 : 1][lane] = zc;
    }
  }
  // which kinds of TF/SF weights occur in the wave
  bool twy = false, twz = false, twx = false;
  if constexpr (TF) {
    twy = __builtin_amdgcn_ballot_w64((fz & 0x3f000000) != 0) != 0;
    twz = __builtin_amdgcn_ballot_w64((fz & 0x00ffffff) != 0) != 0;
    twx = __builtin_amdgcn_ballot_w64((fi & 0x3fc00) != 0) != 0;
  }
  bool special0 = false, dwave = false;  // dwave: rows and columns that meet the design box
  if constexpr (UP) {
    special0 = A.mt.table[0].special != 0;
    const bool in = act && j >= A.mt.d_j0 && j < A.mt.d_j0 + A.mt.d_nj && k + NV > A.mt.d_k0 &&
                    k < A.mt.d_k0 + A.mt.d_nk;
    dwave = A.mt.d_on && __builtin_amdgcn_ballot_w64(in) != 0;
  }

  float one = 1.0f;
  if constexpr (HALF) asm volatile("" : "+s"(one));
  if (XZ && xwave) {
#pragma unroll
    for (int q = 0; q < 3; q++) {
      zone(qy[q], CS + 1, plane(p0 - OWN + q), 0);
      zone(qz[q], CS + 2, plane(p0 - OWN + q), 0);
    }
  }

#pragma nounroll
  for (int i = p0; i < p1; i++) {
    const int pn = plane(i + LEAD);
    const Plane<AD> bx = at(i, CS), bz = at(i, CS + 2);
    // loads of this plane
    qy[3] = ldw<STORE, XZ>(at(pn, CS + 1), own, A.isrc[1]);
    qz[3] = ldw<STORE, XZ>(at(pn, CS + 2), own, A.isrc[2]);
    V x = ldw<STORE, XZ>(bx, own, A.isrc[0]);
    S xl[2] = {}, xh[2] = {}, yl[2] = {}, yh[2] = {};
    if constexpr (GEN) {
      const Plane<AD> by = at(i, CS + 1);
      if (zlo) {
#pragma unroll
        for (int t = 0; t < OWN; t++) {
          xl[t] = ldw1<STORE, XZ>(bx, ol[t], A.isrc[0]);
          yl[t] = ldw1<STORE, XZ>(by, ol[t], A.isrc[1]);
        }
      }
      if (zhi) {
#pragma unroll
        for (int t = 0; t < LEAD; t++) {
          xh[t] = ldw1<STORE, XZ>(bx, oh[t], A.isrc[0]);
          yh[t] = ldw1<STORE, XZ>(by, oh[t], A.isrc[1]);
        }
      }
    }
    V x0 = ldw<STORE, XZ>(bx, r0, A.isrc[0]);
    V x1 = ldw<STORE, XZ>(bx, r1, A.isrc[0]);
    V x2 = ldw<STORE, XZ>(bx, r2, A.isrc[0]);
    V z0 = ldw<STORE, XZ>(bz, r0, A.isrc[2]);
    V z1 = ldw<STORE, XZ>(bz, r1, A.isrc[2]);
    V z2 = ldw<STORE, XZ>(bz, r2, A.isrc[2]);
    const Plane<AD> wx = at(i, CD), wy = at(i, CD + 1), wz = at(i, CD + 2);
    unsigned cls = 0;  // class bytes of the cells
    if constexpr (UP) {
      if (i >= A.mt.cx0 && i < A.mt.cx1) {
        cls = ldt<unsigned>(span<AD>(A.mt.cls, (long long)i * A.sx, (unsigned long long)A.sx + NV), act ? cell : OUT);
        if (GEN && nv < NV) cls &= (1u << (8 * nv)) - 1u;
      }
    }
    V d0 = ldw<STORE, XZ>(wx, own, A.idst[0]);
    V d1 = ldw<STORE, XZ>(wy, own, A.idst[1]);
    V d2 = ldw<STORE, XZ>(wz, own, A.idst[2]);
    // psi of the plane's slab cells: z, and of the x slab or the y slab (a
    // wave in both loads the y slab's where it needs it)
    const int xsl = A.pml ? slab_index(i, nx, A.plo[0], A.phi[0]) : -1;
    F pz0, pz1, pe0, pe1;
    // psi of this plane, slot s: of the z slab (from kFront floats before it), the x slab, the y slab
    auto psiz = [&](int t) {
      return span<AD>(A.psi[2][t], ((long long)i * A.ny * Pz - (int)kFront) * 4,
                      ((unsigned long long)A.ny * Pz + 2 * kFront) * 4);
    };
    auto psix = [&](int t) {
      return span<AD>(A.psi[0][t], (long long)xsl * A.sx * 4, ((unsigned long long)A.sx + NV) * 4);
    };
    const int Py = A.plo[1] + A.phi[1];
    auto psiy = [&](int t) {
      return span<AD>(A.psi[1][t], (long long)i * Py * nz * 4, ((unsigned long long)Py * nz + NV) * 4);
    };
    const O ox = act ? cell * 4u : OUT;
    if (zslab && zm != 0) {
      pz0 = ldt<F>(psiz(0), oz);
      pz1 = ldt<F>(psiz(1), oz);
    }
    float bx_ = 0.f, cx_ = 0.f;
    if (xsl >= 0) {
      using CoefK = __attribute__((address_space(4))) const float;
      bx_ = ((const CoefK*)A.b[0])[i];
      cx_ = ((const CoefK*)A.c[0])[i];
    }
    // Split layer: the stored parts of the lane's cells, in a wave that meets a
    // slab, loaded and stored as whole chunks beside the fields.  (Part by part
    // and cell by cell, behind a branch each, the 12 loads and the coefficients
    // were a chain: 40.4 us a step at 117x110x103, 30.3 so.)
    const bool sany = SP && (zwave || ywave || xsl >= 0);
    F pn0 = {}, pn1 = {}, pn2 = {};
    auto stored = [&](int t) {
      return span<AD>(A.p2[t], (long long)i * A.sx * 4, ((unsigned long long)A.sx + NV) * 4);
    };
    const O op = xsl >= 0 || sy || zm != 0 ? ox : OUT;
    if (sany) {
      pn0 = ldt<F>(stored(0), op);
      pn1 = ldt<F>(stored(1), op);
      pn2 = ldt<F>(stored(2), op);
    }
    if (!SP && xsl >= 0) {
      pe0 = ldt<F>(psix(0), ox);
      pe1 = ldt<F>(psix(1), ox);
    } else if (!SP && ywave) {
      pe0 = ldt<F>(psiy(0), oy);
      pe1 = ldt<F>(psiy(1), oy);
    }
    if constexpr (XZ) {
      if (xwave && (A.per[0] || (i + 2 >= A.xz.i0 && i - 2 < A.xz.i1))) {
        zone(qy[3], CS + 1, pn, 0);
        zone(qz[3], CS + 2, pn, 0);
        zone(x, CS, i, 0);
        zone(x0, CS, i, UP ? -1 : -2);
        zone(x1, CS, i, UP ? 1 : -1);
        zone(x2, CS, i, UP ? 2 : 1);
        zone(z0, CS + 2, i, UP ? -1 : -2);
        zone(z1, CS + 2, i, UP ? 1 : -1);
        zone(z2, CS + 2, i, UP ? 2 : 1);
        zone(d0, CD, i, 0);
        zone(d1, CD + 1, i, 0);
        zone(d2, CD + 2, i, 0);
        if (zlo) {
#pragma unroll
          for (int t = 0; t < OWN; t++) {
            zone1(xl[t], CS, i, k - OWN + t);
            zone1(yl[t], CS + 1, i, k - OWN + t);
          }
        }
        if (zhi) {
          const int ke = zlast ? nz : k + NV;
#pragma unroll
          for (int t = 0; t < LEAD; t++) {
            zone1(xh[t], CS, i, ke + t);
            zone1(yh[t], CS + 1, i, ke + t);
          }
        }
      }
    }
    // this plane's fold factors, and whether a pair of them is zero throughout
    float fu[6] = {};
    if (TF && A.fold) {
      using FoldK = __attribute__((address_space(4))) const float;
      const FoldK* fp = (const FoldK*)(A.fold + (long long)kFoldStride * (1 + i));
#pragma unroll
      for (int t = 0; t < 6; t++) fu[t] = fp[t];
    }
    auto on = [&](int a, int b) { return ((__float_as_uint(fu[a]) | __float_as_uint(fu[b])) << 1) != 0; };
    auto putf = [&](Plane<AD> p, O o, F v) {  // the chunk's cells inside the grid
      if (!GEN || nv == NV) {
        stt(p, o, v);
      } else {
#pragma unroll
        for (int q = 0; q < NV - 1; q++)
          if (q < nv) stt<float>(p, o + 4u * q, v[q]);
      }
    };
    // The derivatives d<axis><component>, each with its TF/SF term and the
    // layer's part.  (2,4) samples a, b, c, e of a stencil.
    auto diff = [&](V a, V b, V c, V e, float r) {
      F d;
#pragma unroll
      for (int q = 0; q < NV; q++) d[q] = r * d24<S>(a[q], b[q], c[q], e[q], one);
      return d;
    };
    // along z: the neighbours come from the adjacent lanes; a row's end takes
    // the cells beyond it (zero, or on a periodic axis the row's first)
    auto diffz = [&](V v, const S* lo, S* hi, float r) {
      S e[NV + 3];
      if constexpr (GEN) {
        if (A.sw.rag && zlast && nv < NV) {
#pragma unroll
          for (int t = 0; t < LEAD; t++)
#pragma unroll
            for (int q = 1; q < NV; q++)
              if (q == nv + t) v[q] = hi[t];
          if (UP && nv == NV - 1) hi[0] = hi[LEAD - 1];
        }
      }
      around<UP, S>(v, e);
      const bool first = GEN ? zlo : zfirst, last = GEN ? zhi : zlast;
#pragma unroll
      for (int t = 0; t < OWN; t++) e[t] = first ? (GEN ? lo[t] : (S)0.f) : e[t];
#pragma unroll
      for (int t = 0; t < LEAD; t++) e[OWN + NV + t] = last ? (GEN ? hi[t] : (S)0.f) : e[OWN + NV + t];
      F d;
#pragma unroll
      for (int q = 0; q < NV; q++) d[q] = r * d24<S>(e[q], e[q + 1], e[q + 2], e[q + 3], one);
      return d;
    };
    int f1 = fz, f2 = fi;  // opaque: unpacked in the branches that need them, not held unpacked along the march
    if constexpr (TF) asm volatile("" : "+v"(f1), "+v"(f2));
    F dxz = diff(qz[0], qz[1], qz[2], qz[3], A.rd[0][2]);
    F dxy = diff(qy[0], qy[1], qy[2], qy[3], A.rd[0][1]);
    if constexpr (TF) {
      if (twx && on(3, 4)) {
#pragma unroll
        for (int q = 0; q < NV; q++) {
          dxz[q] = __builtin_fmaf(fold_b(f2, 10 + q), fu[3], dxz[q]);
          dxy[q] = __builtin_fmaf(fold_b(f2, 14 + q), fu[4], dxy[q]);
        }
      }
    }
    if (!SP && xsl >= 0) {  // x axis: slot 0 = y component (D_x z), slot 1 = z component (D_x y)
#pragma unroll
      for (int q = 0; q < NV; q++) {
        pe0[q] = __builtin_fmaf(cx_, dxz[q], bx_ * pe0[q]);
        pe1[q] = __builtin_fmaf(cx_, dxy[q], bx_ * pe1[q]);
        dxz[q] += pe0[q];
        dxy[q] += pe1[q];
      }
      if (act) {
        putf(psix(0), ox, pe0);
        putf(psix(1), ox, pe1);
      }
      if (ywave) {
        pe0 = ldt<F>(psiy(0), oy);
        pe1 = ldt<F>(psiy(1), oy);
      }
    }
    F dzx = diffz(x, xl, xh, A.rd[2][0]);
    F dzy = diffz(qy[OWN], yl, yh, A.rd[2][1]);
    if constexpr (TF) {
      if (twz && on(1, 2)) {
        const float y1 = fold_b(f2, 0) * fu[1], y2 = fold_b(f2, 1) * fu[2];
#pragma unroll
        for (int q = 0; q < NV; q++) {
          const float w = fold_f(f1, 6 * q);
          dzy[q] = __builtin_fmaf(w, y1, dzy[q]);
          dzx[q] = __builtin_fmaf(w, y2, dzx[q]);
        }
      }
    }
    if (zslab) {
      if (zm != 0) {  // z axis: slot 0 = x component (D_z y), slot 1 = y component (D_z x)
        const F b = lcoef[0][lane], c = lcoef[SP ? 0 : 1][lane];
#pragma unroll
        for (int q = 0; q < NV; q++) {
          pz0[q] = cpml(pz0[q], b[q], c[q], dzy[q]);
          pz1[q] = cpml(pz1[q], b[q], c[q], dzx[q]);
          const bool in = (zm >> q) & 1u;
          dzy[q] = in ? dzy[q] + pz0[q] : dzy[q];
          dzx[q] = in ? dzx[q] + pz1[q] : dzx[q];
        }
        const bool all = zm == (1u << NV) - 1u;
        stt(psiz(0), all ? oz : OUT, pz0);
        stt(psiz(1), all ? oz : OUT, pz1);
        if (!all) {
#pragma unroll
          for (int q = 0; q < NV; q++)
            if ((zm >> q) & 1u) {
              stt<float>(psiz(0), oz + 4u * q, pz0[q]);
              stt<float>(psiz(1), oz + 4u * q, pz1[q]);
            }
        }
      }
    } else if (!SP && zwave) {
      if (zm != 0) {
        const ArgsK* C = again();
        const long long b = ((long long)i * A.ny + j) * Pz;
        float* const a0 = C->psi[2][0] + b;
        float* const a1 = C->psi[2][1] + b;
        const float* const bb = C->b[2] + k;
        const float* const cc = C->c[2] + k;
#pragma unroll
        for (int q = 0; q < NV; q++) {
          if ((zm >> q) & 1u) {
            const int zq = slab_index(k + q, nz, A.plo[2], A.phi[2]);
            const float v0 = cpml(a0[zq], bb[q], cc[q], dzy[q]), v1 = cpml(a1[zq], bb[q], cc[q], dzx[q]);
            a0[zq] = v0;
            a1[zq] = v1;
            dzy[q] += v0;
            dzx[q] += v1;
          }
        }
      }
    }
    F dyx = UP ? diff(x0, x, x1, x2, A.rd[1][0]) : diff(x0, x1, x, x2, A.rd[1][0]);
    F dyz = UP ? diff(z0, qz[OWN], z1, z2, A.rd[1][2]) : diff(z0, z1, qz[OWN], z2, A.rd[1][2]);
    if constexpr (TF) {
      if (twy && on(0, 5)) {
        const float w = fold_f(f1, 24);
#pragma unroll
        for (int q = 0; q < NV; q++) {
          dyz[q] = __builtin_fmaf(fold_b(f2, 2 + q) * w, fu[0], dyz[q]);
          dyx[q] = __builtin_fmaf(fold_b(f2, 6 + q) * w, fu[5], dyx[q]);
        }
      }
    }
    if (!SP && ywave) {
      if (ysl >= 0) {  // y axis: slot 0 = z component (D_y x), slot 1 = x component (D_y z)
#pragma unroll
        for (int q = 0; q < NV; q++) {
          pe0[q] = cpml(pe0[q], by, cy, dyx[q]);
          pe1[q] = cpml(pe1[q], by, cy, dyz[q]);
          dyx[q] += pe0[q];
          dyz[q] += pe1[q];
        }
        putf(psiy(0), oy, pe0);
        putf(psiy(1), oy, pe1);
      }
    }
    // old values
    F o0, o1, o2;
#pragma unroll
    for (int q = 0; q < NV; q++) {
      o0[q] = HALF ? __builtin_fmaf((float)d0[q], A.idst[0], 0.0f) : (float)d0[q];
      o1[q] = HALF ? __builtin_fmaf((float)d1[q], A.idst[1], 0.0f) : (float)d1[q];
      o2[q] = HALF ? __builtin_fmaf((float)d2[q], A.idst[2], 0.0f) : (float)d2[q];
    }
    F n0, n1, n2;
    // new values of cell q from the factor of its curl: -dt, or dt / eps
    auto upd = [&](int q, float k0, float k1, float k2) {
      if constexpr (SP) {  // the two curl terms apart, as off the slab (k1, k2) = (1, 1)
        n0[q] = mulr(-k0, dzy[q]) + (mulr(k0, dyz[q]) + o0[q]);
        n1[q] = mulr(-k1, dxz[q]) + (mulr(k1, dzx[q]) + o1[q]);
        n2[q] = mulr(-k2, dyx[q]) + (mulr(k2, dxy[q]) + o2[q]);
      } else {
        n0[q] = __builtin_fmaf(k0, dyz[q] - dzy[q], o0[q]);
        n1[q] = __builtin_fmaf(k1, dzx[q] - dxz[q], o1[q]);
        n2[q] = __builtin_fmaf(k2, dxy[q] - dyx[q], o2[q]);
      }
    };
    // split field: x component (y, z), y (z, x), z (x, y); the stored parts pn
    auto split = [&](int q, float k0, float k1, float k2) {
      const float k1x = xsl >= 0 ? bx_ : 1.f, k2x = xsl >= 0 ? cx_ : 1.f;
      const float k1y = sy ? by : 1.f, k2y = sy ? cy : 1.f;
      const bool zin = (zm >> q) & 1u;
      const float k1z = zin ? zb[q] : 1.f, k2z = zin ? zc[q] : 1.f;
      auto part = [&](float& stored, float f0, float k1a, float k2a, float ua, float k1b, float k2b, float ub,
                      float n) -> float {
        const float p2 = stored, p1 = f0 - p2;
        const float m1 = __builtin_fmaf(k2a, ua, k1a * p1), m2 = __builtin_fmaf(k2b, ub, k1b * p2);
        const bool out = k2a == 1.0f && k2b == 1.0f;  // outside every slab of the component
        stored = out ? p2 : m2;
        return out ? n : m1 + m2;
      };
      float s0 = pn0[q], s1 = pn1[q], s2 = pn2[q];
      n0[q] = part(s0, o0[q], k1y, k2y, k0 * dyz[q], k1z, k2z, -k0 * dzy[q], n0[q]);
      n1[q] = part(s1, o1[q], k1z, k2z, k1 * dzx[q], k1x, k2x, -k1 * dxz[q], n1[q]);
      n2[q] = part(s2, o2[q], k1x, k2x, k2 * dxy[q], k1y, k2y, -k2 * dyx[q], n2[q]);
      pn0[q] = s0;
      pn1[q] = s1;
      pn2[q] = s2;
    };
    const unsigned in = act ? (1u << nv) - 1u : 0u;
    unsigned put = in;  // cells whose new value this sweep stores
    bool mixed = false;
    if constexpr (UP) {
      const bool dpl = dwave && i >= A.mt.d_i0 && i < A.mt.d_i0 + A.mt.d_ni;
      mixed = __builtin_amdgcn_ballot_w64(cls != 0) != 0 || special0 || dpl;
      if (mixed) {
        // Cells of another class than 0, of the design box, or finished by k_ade.
        // The entries of several cells are loaded together: cell by cell, behind
        // a branch each, the E sweep with a sphere of radius 40 took 72 us at
        // 200^3, 65 so (four at a time; half storage has registers for two:
        // 512x256x256 190 and 183).
        const ArgsK* C = again();
        using Entry = unsigned __attribute__((ext_vector_type(4)));  // ClassEntry: inv_eps, then mat and special bytes
        constexpr int AT = STORE == 1 ? 2 : NV;  // entries in registers at a time
#pragma unroll
        for (int q0 = 0; q0 < NV; q0 += AT) {
          Entry ce[AT];
#pragma unroll
          for (int t = 0; t < AT; t++)
            ce[t] = *reinterpret_cast<const Entry*>(C->mt.table + ((cls >> (8 * (q0 + t))) & 0xffu));
          unsigned over = 0;
          if (dpl) {
#pragma unroll
            for (int t = 0; t < AT; t++) {
              const int dj = j - C->mt.d_j0, dk = k + q0 + t - C->mt.d_k0;
              if (((in >> (q0 + t)) & 1u) && dj >= 0 && dj < C->mt.d_nj && dk >= 0 && dk < C->mt.d_nk) {
                ce[t][0] = ce[t][1] = ce[t][2] = __float_as_uint(
                    C->mt.d_inv_eps[((long long)(i - C->mt.d_i0) * C->mt.d_nj + dj) * C->mt.d_nk + dk]);
                over |= 1u << t;
              }
            }
          }
#pragma unroll
          for (int t = 0; t < AT; t++) {
            const int q = q0 + t;
            const float k0 = C->dt * __uint_as_float(ce[t][0]), k1 = C->dt * __uint_as_float(ce[t][1]),
                        k2 = C->dt * __uint_as_float(ce[t][2]);
            upd(q, k0, k1, k2);
            if (sany && ((in >> q) & 1u)) split(q, k0, k1, k2);
          }
          if (C->ade.on) {
#pragma unroll
            for (int t = 0; t < AT; t++) {
              const int q = q0 + t;
              if (!((in >> q) & 1u) || (ce[t][3] >> 24) == 0 || ((over >> t) & 1u)) continue;
              const long long bq = (long long)(i - C->ade.i0) * C->ade.bsx + (long long)(j - C->ade.j0) * C->ade.bsy +
                                   (k + q - C->ade.k0);  // its curl, for k_ade
              C->ade.curl[0][bq] = dyz[q] - dzy[q];
              C->ade.curl[1][bq] = dzx[q] - dxz[q];
              C->ade.curl[2][bq] = dxy[q] - dyx[q];
              put &= ~(1u << q);
            }
          }
        }
      }
    }
    if (!mixed) {
      const float dt = A.dt;
      float k0 = -dt, k1 = -dt, k2 = -dt;
      if constexpr (UP) {
        k0 = dt * A.mt.table[0].inv_eps[0];
        k1 = dt * A.mt.table[0].inv_eps[1];
        k2 = dt * A.mt.table[0].inv_eps[2];
      }
#pragma unroll
      for (int q = 0; q < NV; q++) {
        upd(q, k0, k1, k2);
        if (sany && ((in >> q) & 1u)) split(q, k0, k1, k2);
      }
    }
    if (sany && op != OUT) {
      putf(stored(0), op, pn0);
      putf(stored(1), op, pn1);
      putf(stored(2), op, pn2);
    }
    if constexpr (SO) {
      if (i >= A.soft.lo && i < A.soft.hi) {
        const ArgsK* C = again();
        for (int t = 0; t < C->soft.n; t++) {
          if (C->soft.i[t] != i || own != (O)C->soft.cell[t] * ES) continue;
          const int at = C->soft.q[t], comp = C->soft.comp[t];
          const float val = C->soft.val[t];
          auto take = [&](F& v, int c) {
#pragma unroll
            for (int q = 0; q < NV; q++)
              if (comp == c && at == q) v[q] -= val;
          };
          take(n0, 0);
          take(n1, 1);
          take(n2, 2);
        }
      }
    }
    if constexpr (XZ) {
      if (xwave && i >= A.xz.i0 && i < A.xz.i1) {  // new values of zone cells to the FP32 copy too
#pragma unroll
        for (int q = 0; q < NV; q++) {
          if ((put & xm) >> q & 1u) {
            const O o = in_copy(i, j, k + q);
            stt<float>(copy(CD), o, n0[q]);
            stt<float>(copy(CD + 1), o, n1[q]);
            stt<float>(copy(CD + 2), o, n2[q]);
          }
        }
      }
    }
    constexpr unsigned ALL = (1u << NV) - 1u;
    // whole chunks with one store per component for every lane (a lane that
    // stores only some cells addresses none here), so that the number of
    // stores in flight is known and, in E, the wait for the next plane's loads
    // does not reach them.  (In H the loop's head waits for all that is under way,
    // these stores too: on the first way in that is the queues.)
    const O whole = put == ALL ? own : OUT;
    using H = Vec<Word<STORE, false>, NV>;
    auto word = [&](F v, float sc) {
      H h;
#pragma unroll
      for (int q = 0; q < NV; q++) h[q] = (Word<STORE, false>)(STORE == 0 ? v[q] : __builtin_fmaf(v[q], sc, 0.0f));
      return h;
    };
    const H h0 = word(n0, A.sdst[0]), h1 = word(n1, A.sdst[1]), h2 = word(n2, A.sdst[2]);
    stt(wx, whole, h0);
    stt(wy, whole, h1);
    stt(wz, whole, h2);
    if (put != ALL && put != 0) {
#pragma unroll
      for (int q = 0; q < NV; q++)
        if ((put >> q) & 1u) {
          stt<Word<STORE, false>>(wx, own + ES * q, h0[q]);
          stt<Word<STORE, false>>(wy, own + ES * q, h1[q]);
          stt<Word<STORE, false>>(wz, own + ES * q, h2[q]);
        }
    }
#pragma unroll
    for (int q = 0; q < 3; q++) {
      qy[q] = qy[q + 1];
      qz[q] = qz[q + 1];
    }
  }
}

// ------------------------------------------------------------ launcher
namespace {

template <typename K>
int resident_waves(K kernel) {  // waves of one launch that fit on the device at once
  int dev = 0, per = 0;
  hipDeviceProp_t p;
  if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&p, dev) != hipSuccess) return 3072;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, 64, 0) != hipSuccess || per < 1) per = 1;
  return per * p.multiProcessorCount;
}

template <int UP, int STORE, bool GEN, bool SP, bool TF, bool XZ, int AD, bool SO = false>
void go(SweepArgs& A, hipStream_t st) {
  static const int slots = resident_waves(k_sweep<UP, STORE, GEN, SP, TF, XZ, AD, SO>);
  Sweep& w = A.sw;
  const int len = w.i1 - w.i0, nlb = w.lb1 - w.lb0, nhb = w.hb1 - w.hb0;
  // Segments.  Up to six planes per resident wave: one round of waves, each
  // marching its share (us a step: 64^3 in segments of 1 / 2 / 8 planes 12.7 /
  // 15.4 / 35.4, 128^3 in 1 / 2 / 3 / 5 planes 41.0 / 39.4 / 38.3 / 41.7).
  // Beyond: several rounds of short segments, which balance the planes and
  // rows with a layer against those without; shorter ones load the three
  // planes of a segment's start too often (256^3 in 1 / 2 / 3 / 6 / 8 planes
  // FP32 338 / 311 / 296 / 298 / 310, FP16 251 / 212 / 196 / 192 / 191).
  // A wave takes the rows beside its own from its XCD's L2, where they are only
  // while the waves of these rows march abreast.  So planes larger than what the
  // XCD's waves hold at once run in strips of that size, and segments end before
  // waves drift far apart.  FP32, all steps over the whole grid, without that and
  // so: 512x500x500 2215 (40.8 bytes a cell from beyond L2) and 2039, 512^3 2150
  // and 2043, 300x512x1024 2747 and 2457, 100x1024x1024 1851 and 1690, 400^3 1066
  // and 1001; FP16 512x500x500 1408 and 1190.  Segments of 4 / 6 / 8 / 12 planes
  // there: FP32 2048 / 2039 / 2053 / 2071, FP16 1262 / 1219 / 1221 / 1211; strips of
  // half that size, FP32: 2040 / 2044 / 2069 / 2097.
  const double share = (double)nlb * len / slots;
  w.seg = share <= 6 ? std::max(1, (int)ceil(share))
                     : std::min(std::max(STORE == 1 ? 4 : 2, (int)(share / 6 + 0.5)), STORE == 1 ? 12 : 6);
  const int strips = share <= 6 ? 1 : (nlb * NXCD + slots - 1) / slots;
  A.strip = (nlb + std::max(strips, 1) - 1) / std::max(strips, 1);
  auto segs = [&](int a, int b) { return (long long)((b - a + w.seg - 1) / w.seg); };
  const long long n[3] = {segs(w.i0, w.h0) * nlb, segs(w.h0, w.h1) * (nlb - nhb), segs(w.h1, w.i1) * nlb};
  const long long blocks = n[0] + n[1] + n[2];
  const long long more = (record_threads(A.pr) + 63) / 64;
  // (a launch of 2^32 lanes or more may run only some of its blocks, without an error)
  if (blocks + NXCD + more >= (1LL << 26)) {
    fail_launch("k_sweep", "2^26 blocks or more");
    return;
  }
  w.total[0] = (int)n[0];
  w.total[1] = (int)(n[0] + n[1]);
  w.total[2] = (int)blocks;
  w.per = (w.total[2] + NXCD - 1) / NXCD;
  if (blocks == 0 && more == 0) return;
  hipLaunchKernelGGL((k_sweep<UP, STORE, GEN, SP, TF, XZ, AD, SO>), dim3(w.per * NXCD + (int)more), dim3(64), 0, st, A);
  note_launch(UP ? "k_sweep E" : "k_sweep H");
}

// What the descriptors can span of a plane, of its psi and weights, and of the field set.
int addressing(const SweepArgs& A) {
  if ((unsigned long long)(A.sx + 64) * 4 >= kBytes ||
      ((unsigned long long)A.ny * (A.plo[2] + A.phi[2]) + 64) * 4 >= kBytes ||
      (unsigned long long)A.sw.NL * sizeof(int2) >= kBytes)
    return kHuge;
  return 6 * A.comp >= kBytes ? kFar : kNear;
}

// The variant of a configuration.  The plain ones (no GEN) need rows that fill
// a wave or a whole fraction of it and a z axis without wrap-around; the far
// and huge ones and those of the split layer and the zone are built for the
// general case only.
template <int UP, int STORE, bool XZ>
void pick(SweepArgs& A, bool split, hipStream_t st) {
  Sweep& w = A.sw;
  w.rag = A.nz % NV;
  w.zgap = A.nz - A.phi[2] - A.plo[2];
  if (w.i1 <= w.i0) return;
  const int ad = addressing(A);
  const bool huge = ad == kHuge, far = ad == kFar;
  const bool plain = w.rag == 0 && !A.per[2] && 64 % w.nzv == 0;
  if (huge || (XZ && far)) {
    if (split) go<UP, STORE, true, true, !XZ, XZ, kHuge>(A, st);
    else go<UP, STORE, true, false, !XZ, XZ, kHuge>(A, st);
  } else if constexpr (XZ) {
    if (split) go<UP, STORE, true, true, false, true, kNear>(A, st);
    else go<UP, STORE, true, false, false, true, kNear>(A, st);
  } else if (far) {
    if (split) go<UP, STORE, true, true, true, false, kFar>(A, st);
    else go<UP, STORE, true, false, true, false, kFar>(A, st);
  } else if (split) {
    go<UP, STORE, true, true, true, false, kNear>(A, st);
  } else if (A.soft.n > 0) {  // FP32 E (launch_sweep: soft_in)
    constexpr bool SO = UP && STORE == 0;
    if (plain) go<UP, STORE, false, false, false, false, kNear, SO>(A, st);
    else go<UP, STORE, true, false, false, false, kNear, SO>(A, st);
  } else if (plain) {
    if (A.fold) go<UP, STORE, false, false, true, false, kNear>(A, st);
    else go<UP, STORE, false, false, false, false, kNear>(A, st);
  } else {
    if (A.fold) go<UP, STORE, true, false, true, false, kNear>(A, st);
    else go<UP, STORE, true, false, false, false, kNear>(A, st);
  }
}

template <int STORE>
void fill(SweepArgs& A, int up, bool zone, const Grid& g, const void* fields, const Scales& sc, const Cpml& pm) {
  const Fields<STORE>& f = *static_cast<const Fields<STORE>*>(fields);
  A.set = reinterpret_cast<char*>(f.E[0]);
  A.comp = (unsigned long long)(reinterpret_cast<char*>(f.E[1]) - A.set);
  A.nx = g.nx;
  A.ny = g.ny;
  A.nz = g.nz;
  A.sx = g.sx;
  A.dt = g.dt;
  A.pml = pm.on;
  for (int a = 0; a < 3; a++) {
    A.per[a] = g.per[a];
    for (int c = 0; c < 3; c++)  // (the zone's variants hold converted values)
      A.rd[a][c] = g.rd[a] * (STORE == 1 && !zone ? (up ? sc.ih[c] : sc.ie[c]) : 1.0f);
    A.isrc[a] = up ? sc.ih[a] : sc.ie[a];
    A.idst[a] = up ? sc.ie[a] : sc.ih[a];
    A.sdst[a] = up ? sc.se[a] : sc.sh[a];
    A.plo[a] = pm.plo[a];
    A.phi[a] = pm.phi[a];
    A.b[a] = up ? pm.bE[a] : pm.bH[a];
    A.c[a] = up ? pm.cE[a] : pm.cH[a];
    A.p2[a] = up ? pm.p2E[a] : pm.p2H[a];
    for (int s = 0; s < 2; s++) A.psi[a][s] = up ? pm.psiE[a][s] : pm.psiH[a][s];
  }
  A.xz = sc.xz;
}

}  // namespace

// Weights of the folded TF/SF source (fold_pack) of every chunk, packed by the
// factor they belong to: x bits 0-23 the z weights of its cells, bits 24-29 the
// y weight; y bits 0, 1 the inside flags along y of factors 1 and 2, bits
// 2-5 and 6-9 those along z of factors 0 and 5 for its cells, bits 10-13 and
// 14-17 the flags of factors 3 and 4.
__global__ __launch_bounds__(256) void k_fold_weights(Tfsf tf, int2* out, int ny, int nz, int nzv) {
  const long long idx = blockIdx.x * 256LL + threadIdx.x;
  if (idx >= 2LL * ny * nzv) return;
  const int half = idx >= (long long)ny * nzv;
  const int r = (int)(idx - (half ? (long long)ny * nzv : 0));
  const int j = r / nzv, k = NV * (r - j * nzv);
  const int hd[5] = {tf.hlo[1], tf.hhi[1], tf.hlo[2], tf.hhi[2], tf.sf_inside};
  int fz = 0, fi = 0;
  for (int q = 0; q < NV && k + q < nz; q++) {
    const int w = fold_pack(half, j, k + q, hd);
    const int w0 = w & 63, w1 = (w >> 6) & 63, w2 = (w >> 12) & 63, w5 = (w >> 18) & 63;
    fz |= (w1 | w2) << (6 * q);  // equal where both are set
    fz |= (w0 | w5) << 24;
    fi |= (w1 != 0) | (w2 != 0) << 1 | (w0 != 0) << (2 + q) | (w5 != 0) << (6 + q) | ((w >> 24) & 1) << (10 + q) |
          ((w >> 25) & 1) << (14 + q);
  }
  out[idx] = make_int2(fz, fi);
}

long long fold_weights_size(const Grid& g) { return 2LL * g.ny * ((g.nz + 3) / 4); }

void launch_fold_weights(const Tfsf& tf, int2* out, const Grid& g, hipStream_t st) {
  const long long n = fold_weights_size(g);
  hipLaunchKernelGGL(k_fold_weights, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, tf, out, g.ny, g.nz,
                     (g.nz + 3) / 4);
  note_launch("k_fold_weights");
}

void launch_sweep(int up, int store, const Grid& g, const void* fields, const Scales& sc, const Cpml& pm,
                  const Materials& mt, const Ade& ade, int i0, int i1, const float* fold, const int2* foldw,
                  const Probes* pr, const Soft* soft, hipStream_t st) {
  SweepArgs A{};
  Soft here{};  // the sources of these planes
  for (int t = 0; soft && t < soft->n; t++) {
    if (soft->ijk[t][0] < i0 || soft->ijk[t][0] >= i1) continue;
    here.comp[here.n] = soft->comp[t];
    here.q[here.n] = soft->q[t];
    here.val[here.n] = soft->val[t];
    for (int a = 0; a < 3; a++) here.ijk[here.n][a] = soft->ijk[t][a];
    here.n++;
  }
  if (pr) A.pr = *pr;
  A.fold = fold;
  A.foldw = foldw ? foldw + (up ? fold_weights_size(g) / 2 : 0) : nullptr;
  A.mt = mt;
  A.ade.on = ade.on;
  A.ade.i0 = ade.i0;
  A.ade.j0 = ade.j0;
  A.ade.k0 = ade.k0;
  A.ade.bsx = ade.bsx;
  A.ade.bsy = ade.bsy;
  for (int c = 0; c < 3; c++) A.ade.curl[c] = ade.curl[c];
  const bool split = pm.on && pm.split;
  Sweep& w = A.sw;
  w.nzv = (g.nz + NV - 1) / NV;
  w.NL = (long long)w.nzv * g.ny;
  const int nlb = (int)((w.NL + 63) / 64);
  if (store) fill<1>(A, up, false, g, fields, sc, pm);
  else fill<0>(A, up, false, g, fields, sc, pm);
  // Soft sources are subtracted where E is new by FP32 variants of their own
  // (SO), which only launches with sources run: us a step at 44^3, 100^3, 128^3,
  // 160^3, 198^3 11.2, 23.2, 34.4, 62.5, 101.3 so and 13.1, 24.8, 36, 63.6, 102.2
  // with k_soft's launch after the sweep; from 206^3 on both take the same.  In
  // the one ragged variant that all grids ran before, the block cost those
  // without sources 1% to 4%: 131^3 39.7 and 39.4 without it, 180^3 78.2 and 76.6,
  // 300^3 453 and 432.  With the fold or in half storage it spills more, and
  // every step takes 2 to 4% longer: there k_soft follows.
  const bool soft_in = here.n > 0 && here.n <= kSweepSoft && store == 0 && !fold && !split && addressing(A) == kNear;
  if (soft_in) {
    A.soft.lo = g.nx;
    A.soft.n = here.n;
    for (int t = 0; t < here.n; t++) {
      A.soft.i[t] = here.ijk[t][0];
      A.soft.q[t] = here.ijk[t][2] % NV;
      A.soft.cell[t] = (long long)here.ijk[t][1] * g.nz + here.ijk[t][2] / NV * NV;
      A.soft.comp[t] = here.comp[t];
      A.soft.val[t] = here.val[t];
      A.soft.lo = std::min(A.soft.lo, here.ijk[t][0]);
      A.soft.hi = std::max(A.soft.hi, here.ijk[t][0] + 1);
    }
  }
  // blocks [b0, b1) of the planes [a, b), without the hole set in w
  auto part = [&](int a, int b, int b0, int b1, bool zone) {
    w.i0 = a;
    w.i1 = b;
    w.lb0 = b0;
    w.lb1 = b1;
    if (zone) fill<1>(A, up, true, g, fields, sc, pm);
    if (zone) up ? pick<1, 1, true>(A, split, st) : pick<0, 1, true>(A, split, st);
    else if (store) up ? pick<1, 1, false>(A, split, st) : pick<0, 1, false>(A, split, st);
    else up ? pick<1, 0, false>(A, split, st) : pick<0, 0, false>(A, split, st);
  };
  w.h0 = w.h1 = i1;
  w.hb0 = w.hb1 = nlb;
  if (store == 1 && sc.xz.on) {
    // The blocks whose stencils reach the FP32 zone run the zone's variants,
    // the others the plain ones, which skip those: the two launches write
    // disjoint cells and read only the other family of fields.  (256^3 with a
    // zone of 21^3 cells: the two zone launches take 26 us a step, 121 with zone
    // variants on every block of the zone's planes.)
    const Exact& x = sc.xz;
    w.h0 = g.per[0] ? i0 : std::min(std::max(x.i0 - 3, i0), i1);
    w.h1 = g.per[0] ? i1 : std::min(std::max(x.i1 + 3, w.h0), i1);
    w.hb0 = g.per[1] ? 0 : (int)((long long)std::max(x.j0 - 3, 0) * w.nzv / 64);
    w.hb1 = g.per[1] ? nlb : (int)(((long long)std::min(x.j1 + 3, g.ny) * w.nzv + 63) / 64);
    part(i0, i1, 0, nlb, false);
    A.pr.n = 0;
    const int a = w.h0, b = w.h1, b0 = w.hb0, b1 = w.hb1;
    w.h0 = w.h1 = b;
    w.hb0 = w.hb1 = b1;
    part(a, b, b0, b1, true);
  } else {
    part(i0, i1, 0, nlb, false);
  }
  if (here.n > 0 && !soft_in) launch_soft(store, g, fields, sc, here, st);
}

}  // namespace dtm
