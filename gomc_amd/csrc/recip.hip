// Whole-box reciprocal space: structure factors S(k) of every atom
// (Ewald::BoxReciprocalSums, src/Ewald.cpp:193-406) and the k-space force on
// every atom (Ewald::BoxForceReciprocal, src/Ewald.cpp:1496-1596; the same
// per-atom sums make VirialReciprocal's intramolecular term, 1168-1305), as
// FP64 matrix products on the matrix cores.
//
// The k list is made of columns: all nz = -m..m at one (nx, ny), nx >= 0
// (nz = 1..m at (0, 0)).  With a = e^{i (kx x + ky y)} and z = c + i s =
// e^{i kz |nz| z} the two signs of nz share their products:
//   q e^{i k.r}(+nz) = (ar c - ai s) + i (ai c + ar s)
//   q e^{i k.r}(-nz) = (ar c + ai s) + i (ai c - ar s)
// so S of a column is four real sums over atoms, ar c, ar s, ai c, ai s: a
// matrix product of [2 x columns] x [atoms] by [atoms] x [2 (m + 1)], two
// multiply-adds per (atom, k-vector).  The force on an atom is the transposed
// product: with U, D = pref (R+ +- R-) and V, E = pref (I+ +- I-) of a
// column's nz,
//   sum_nz f = ar G1 + ai G2,  G1 = sum (s D - c V),  G2 = sum (c U + s E)
//   sum_nz nz f = ar H1 + ai H2,  H1 = sum nz (s U - c E),  H2 = sum nz (c D + s V)
// f = im R - re I the k-vector's term; Fx and Fy take nx, ny times the
// first, Fz the second: four multiply-adds per (atom, k-vector).
//
// V_MFMA_F64_16X16X4: lane l holds A[i = l % 16][k = l / 16],
// B[k = l / 16][j = l % 16] and, in register v, D[i = l / 16 + 4 v][j].
#include <algorithm>
#include <cmath>
#include <mutex>
#include <string>
#include <vector>

#include "box.hpp"

namespace gomc {
namespace {

typedef double v4d __attribute__((ext_vector_type(4)));

__device__ __forceinline__ v4d Mfma(double a, double b, v4d c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

constexpr int kMmThreads = 512, kMmWaves = kMmThreads / kWave;
constexpr int kPhaseRun = 8;  // table entries one thread makes: two sincos, then products

// LDS, named as such: a plain pointer into an out-of-line function is a flat
// address.
#define LMEM __attribute__((address_space(3)))

// scale e^{i pi n u} for n = n0 .. n0 + count - 1, stored (re, im) `stride`
// doubles apart: the first from its own argument, the others by complex
// products, so no entry is more than kPhaseRun - 1 products from a sincos.
// u = 2 r / L: in half-turns the reduction of the argument is exact and
// short, where sincos of the angle carries a branch for huge arguments and
// its registers.
__device__ __forceinline__ void PhaseRun(double u, int n0, int count, double scale,
                                         LMEM double *out, int stride) {
  double s1, c1, im, re;
  sincospi(u, &s1, &c1);
  sincospi(double(n0) * u, &im, &re);
  re *= scale;
  im *= scale;
  for (int n = 0; n < count; ++n) {
    out[0] = re;
    out[1] = im;
    out += stride;
    const double nr = fma(re, c1, -(im * s1));
    im = fma(re, s1, im * c1);
    re = nr;
  }
}

__device__ __forceinline__ double2 PhaseOf(double halfTurns) {
  double s, c;
  sincospi(halfTurns, &s, &c);
  return make_double2(c, s);
}

__device__ __forceinline__ LMEM double *Lds(double *p) { return (LMEM double *)p; }

// ------------------------------------------------------ structure factors --
struct SumsArgs {
  const double *x, *y, *z, *q;
  const int *mol;
  int natoms, K;
  const int4 *cols;   // {index of nz = 0, nx, ny, m}; m = -1: padding
  const int4 *units;  // [nB][kMmWaves] {column group of 16, first nz, tiles of 8 nz, 0}
  int nB, chunks, aChunk;
  int E, oy, oz, T;   // table entries per atom, where y and z start, atoms per tile
  int nx, ny, Ez;     // entries 0..nx, 0..ny (-1: no table), Ez of the block's z window
  double ux, uy, uz;  // 2 / L_d
  const double *pref;
  double2 *part;      // [chunks][K] (S_R, S_I)
  double *sumR, *sumI;
  Partial4 *partials;
  unsigned *counter;
  double *result;
};

// One workgroup: eight waves, each a unit of 16 columns x up to 32 nz, over
// one chunk of atoms.  Atoms that carry no charge or sit in the reservoir
// are dropped first (512 tested at a time, kept in order), the rest taken T
// at a time: their per-axis phase tables, the charge in the x phases, go to
// LDS, shared by the eight waves, and a wave makes its A operand q ex ey on
// the fly from two table reads (5 FP64 operations for 4 atoms x 16 columns
// against up to 8 MFMAs).  A tile is padded to whole steps of 4 atoms by
// charge 0.  Bound by the matrix cores and the table builds between them:
// 10,000 waters (30,000 atoms, K = 30,902, 5.8 GFLOP with the padding of
// 16-column, 8-nz tiles) 159 us, 36 TFLOP/s; 620 us as one rotating phase
// per (atom, k-vector) on the vector units.
template <bool direct>  // no x and y tables: a very long box
__global__ void __launch_bounds__(kMmThreads, 4) RecipSumsPartKernel(const SumsArgs a) {
  extern __shared__ double2 tab[];
  __shared__ int list[kMmThreads];
  __shared__ int wcnt[kMmWaves];
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int g = blockIdx.x % a.nB, chunk = blockIdx.x / a.nB;
  const int4 unit = a.units[g * kMmWaves + wave];
  const int group = __builtin_amdgcn_readfirstlane(unit.x);
  const int w0 = __builtin_amdgcn_readfirstlane(unit.y);  // the same in the block's units
  const int nt = __builtin_amdgcn_readfirstlane(unit.z);
  const int4 col = a.cols[group * 16 + lane % 16];
  const double sy = col.z < 0 ? -1.0 : 1.0;
  v4d accR[4], accI[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) accR[t] = accI[t] = v4d{0.0, 0.0, 0.0, 0.0};
  const int segX = direct ? 0 : (a.nx + kPhaseRun) / kPhaseRun,
            segY = direct ? 0 : (a.ny + kPhaseRun) / kPhaseRun, segs = segX + segY + a.Ez / kPhaseRun;
  const int a0 = min(a.natoms, chunk * a.aChunk), a1 = min(a.natoms, a0 + a.aChunk);
  for (int base = a0; base < a1; base += kMmThreads) {
    __syncthreads();  // the previous batch's list is read
    const int i = base + tid;
    bool keep = false;
    if (i < a1) keep = a.mol[i] >= 0 && !(fabs(a.q[i]) < 0.000000001);
    const uint64_t mask = __ballot(keep);
    if (lane == 0) wcnt[wave] = __popcll(mask);
    __syncthreads();
    int off = 0, n = 0;
    for (int w = 0; w < kMmWaves; ++w) {
      if (w < wave) off += wcnt[w];
      n += wcnt[w];
    }
    if (keep) list[off + __popcll(mask & ((uint64_t(1) << lane) - 1))] = i;
    for (int tile = 0; tile < n; tile += a.T) {
      const int tn = (min(a.T, n - tile) + 3) & ~3;
      __syncthreads();  // the list is written, the previous tile's tables read
      for (int it = tid; it < tn * segs; it += kMmThreads) {
        const int s = it / tn, at = it - s * tn;
        const bool real = tile + at < n;
        const int j = list[min(tile + at, n - 1)];
        LMEM double *row = Lds(reinterpret_cast<double *>(tab + size_t(at) * a.E));
        if (s < segX) {
          const int n0 = s * kPhaseRun;
          PhaseRun(a.ux * a.x[j], n0, min(kPhaseRun, a.nx + 1 - n0), real ? a.q[j] : 0.0,
                   row + 2 * n0, 2);
        } else if (s < segX + segY) {
          const int n0 = (s - segX) * kPhaseRun;
          PhaseRun(a.uy * a.y[j], n0, min(kPhaseRun, a.ny + 1 - n0), 1.0, row + 2 * (a.oy + n0), 2);
        } else {
          const int n0 = (s - segX - segY) * kPhaseRun;
          PhaseRun(a.uz * a.z[j], w0 + n0, kPhaseRun, 1.0, row + 2 * (a.oz + n0), 2);
        }
      }
      __syncthreads();
      if (nt > 0) {
        const double2 *row = tab + size_t(lane / 16) * a.E;
        const double2 *px = row + col.y, *py = row + a.oy + abs(col.z);
        const double *zr = reinterpret_cast<const double *>(row + a.oz) + lane % 16;
        const int step = 4 * a.E;
        for (int s = 0; s < tn; s += 4, px += step, py += step, zr += 2 * step) {
          double ar, ai;
          if constexpr (!direct) {
            const double2 ex = *px, ey = *py;
            const double eyi = sy * ey.y;
            ar = fma(ex.x, ey.x, -(ex.y * eyi));
            ai = fma(ex.x, eyi, ex.y * ey.x);
          } else {
            const int at = tile + s + lane / 16, j = list[min(at, n - 1)];
            const double2 p = PhaseOf(col.y * (a.ux * a.x[j]) + col.z * (a.uy * a.y[j]));
            const double q = at < n ? a.q[j] : 0.0;
            ar = q * p.x;
            ai = q * p.y;
          }
#pragma unroll
          for (int t = 0; t < 4; ++t)
            if (t < nt) {
              const double b = zr[16 * t];
              accR[t] = Mfma(ar, b, accR[t]);
              accI[t] = Mfma(ai, b, accI[t]);
            }
        }
      }
    }
  }
  // lane pairs (c, s) of one nz: the even lane writes S(+nz), the odd S(-nz)
  double2 *out = a.part + size_t(chunk) * a.K;
  const bool odd = lane & 1;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int4 cv = a.cols[group * 16 + lane / 16 + 4 * v];
    const int lo = (cv.y == 0 && cv.z == 0) ? 1 : -cv.w;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const double pR = accR[t][v], pI = accI[t][v];  // even: ar c, ai c; odd: ar s, ai s
      const double oR = __shfl_xor(pR, 1), oI = __shfl_xor(pI, 1);
      const int nz = w0 + 8 * t + (lane % 16) / 2;
      if (t < nt && nz <= cv.w) {
        if (!odd && nz >= lo) out[cv.x + nz] = make_double2(pR - oI, pI + oR);
        if (odd && nz > 0 && -nz >= lo) out[cv.x - nz] = make_double2(oR + pI, oI - pR);
      }
    }
  }
}

// The chunks' sums of every k-vector added (slice s of four takes chunks s,
// s + 4, ..., then the slices in order), and the energy pref (R^2 + I^2).
constexpr int kSumsSlices = 4;

__global__ void __launch_bounds__(kBlock) RecipSumsKernel(const SumsArgs a) {
  __shared__ double red[kBlock / kWave];
  __shared__ double2 sl[kSumsSlices][kWave];
  const int lane = threadIdx.x % kWave, s = threadIdx.x / kWave;
  const int k = blockIdx.x * kWave + lane;
  double2 v = make_double2(0.0, 0.0);
  if (k < a.K)
#pragma unroll 8
    for (int c = s; c < a.chunks; c += kSumsSlices) {
      const double2 p = a.part[size_t(c) * a.K + k];
      v.x += p.x;
      v.y += p.y;
    }
  sl[s][lane] = v;
  __syncthreads();
  double e = 0.0;
  if (s == 0 && k < a.K) {
    for (int i = 1; i < kSumsSlices; ++i) {
      v.x += sl[i][lane].x;
      v.y += sl[i][lane].y;
    }
    a.sumR[k] = v.x;
    a.sumI[k] = v.y;
    e = (v.x * v.x + v.y * v.y) * a.pref[k];
  }
  Partial4 part{0, 0, 0, 0};
  part.recip = BlockSum(e, red);
  FinishPartials(part, a.partials, a.counter, a.result);
}

// ------------------------------------------------------------------ force --
// The coefficients of the four sums of every column, as the A operands of
// the force product: column groups of 4, row i = column + 4 (G1, G2, H1, H2),
// depth 4 per step = (c, s) of two nz.
struct CoefArgs {
  const int4 *cols;
  const int *fstart;  // [ngrp + 1] first step of each group
  int ngrp, steps, K;
  const double *pref, *sumR, *sumI;
  double *coef;       // [steps][64]
};

__global__ void __launch_bounds__(kBlock) RecipCoefKernel(const CoefArgs a) {
  const int step = blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave, lane = threadIdx.x % kWave;
  if (step >= a.steps) return;
  int lo = 0, hi = a.ngrp;  // the group holding this step
  while (hi - lo > 1) {
    const int mid = (lo + hi) / 2;
    if (a.fstart[mid] <= step) lo = mid;
    else hi = mid;
  }
  const int4 col = a.cols[lo * 4 + lane % 4];
  const int type = (lane % 16) / 4, kk = lane / 16;
  const int nz = 2 * (step - a.fstart[lo]) + kk / 2;
  const bool s = kk & 1;
  const int first = (col.y == 0 && col.z == 0) ? 1 : -col.w;
  double rp = 0.0, ip = 0.0, rm = 0.0, im = 0.0;
  if (nz <= col.w) {
    if (nz >= first) {
      const int k = col.x + nz;
      rp = a.pref[k] * a.sumR[k];
      ip = a.pref[k] * a.sumI[k];
    }
    if (nz > 0 && -nz >= first) {
      const int k = col.x - nz;
      rm = a.pref[k] * a.sumR[k];
      im = a.pref[k] * a.sumI[k];
    }
  }
  const double U = rp + rm, D = rp - rm, V = ip + im, Ee = ip - im;
  double v;
  if (type == 0) v = s ? D : -V;
  else if (type == 1) v = s ? Ee : U;
  else if (type == 2) v = nz * (s ? U : -Ee);
  else v = nz * (s ? V : D);
  a.coef[size_t(step) * kWave + lane] = v;
}

struct ForceArgs {
  const double *x, *y, *z, *q;
  int natoms;
  const int4 *cols;
  const int *fstart;
  int ngrp, chunks;
  int nx, ny;        // table entries 0..nx, 0..ny
  int zSteps, maxSteps;  // steps per z window, of the longest column
  double cx, cy, cz;  // 2 pi / L_d
  double ux, uy, uz;  // 2 / L_d
  const double *coef;
  double *part;      // [chunks][xyz][natoms]: 2 q sum_k f k_d
};

// One workgroup: 16 NT atoms, eight waves over the column groups of one
// chunk (wave w of chunk c takes groups c + chunks (w + 8 i); groups are
// sorted by length, so the waves' shares are alike).  B operands, the z
// phases of the atoms, and the x and y phases sit in LDS; an A operand is
// one 8-byte read per lane for NT MFMAs.  Bound by the matrix cores on a
// large box: 188 us on 10,000 waters (8.3 GFLOP with the padding), 44 TFLOP/s;
// 635 us as six multiply-adds and a complex product per (atom, k-vector) on
// the vector units.  1000 waters 9.8 us, before 16.4.
template <int NT, bool XY>  // XY: x and y phases from tables
__global__ void __launch_bounds__(kMmThreads, 4) RecipForcePartKernel(const ForceArgs a) {
  constexpr int A = 16 * NT;
  extern __shared__ double2 tab[];
  __shared__ double red[kMmWaves][3][A];
  double2 *tx = tab, *ty = tx + (XY ? (a.nx + 1) * A : 0);
  double *tz = reinterpret_cast<double *>(ty + (XY ? (a.ny + 1) * A : 0));
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int chunk = blockIdx.x % a.chunks, a0 = blockIdx.x / a.chunks * A;
  const int segX = XY ? (a.nx + kPhaseRun) / kPhaseRun : 0,
            segY = XY ? (a.ny + kPhaseRun) / kPhaseRun : 0;
  for (int it = tid; it < A * (segX + segY); it += kMmThreads) {
    const int at = it % A, s = it / A, j = min(a0 + at, a.natoms - 1);
    const bool isX = s < segX;
    const int n0 = (isX ? s : s - segX) * kPhaseRun;
    PhaseRun(isX ? a.ux * a.x[j] : a.uy * a.y[j], n0,
             min(kPhaseRun, (isX ? a.nx : a.ny) + 1 - n0), 1.0,
             Lds(reinterpret_cast<double *>((isX ? tx : ty) + n0 * A + at)), 2 * A);
  }
  double fx[NT], fy[NT], fz[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) fx[t] = fy[t] = fz[t] = 0.0;
  const int kk = lane / 16, jj = lane % 16;
  for (int w0 = 0; w0 < a.maxSteps; w0 += a.zSteps) {
    const int nw = min(a.zSteps, a.maxSteps - w0);  // steps of this window, 2 nz each
    __syncthreads();
    for (int it = tid; it < A * ((2 * nw + kPhaseRun - 1) / kPhaseRun); it += kMmThreads) {
      const int at = it % A, n0 = it / A * kPhaseRun, j = min(a0 + at, a.natoms - 1);
      PhaseRun(a.uz * a.z[j], 2 * w0 + n0, min(kPhaseRun, 2 * nw - n0), 1.0,
               Lds(tz + (n0 * A + at) * 2), 2 * A);
    }
    __syncthreads();
    for (int g = chunk + a.chunks * wave; g < a.ngrp; g += a.chunks * kMmWaves) {
      const int f0 = a.fstart[g];
      const int ns = min(a.fstart[g + 1] - f0 - w0, nw);
      if (ns <= 0) break;  // groups get no longer
      const int4 col = a.cols[g * 4 + kk];
      v4d acc[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = v4d{0.0, 0.0, 0.0, 0.0};
      const double *cf = a.coef + size_t(f0 + w0) * kWave + lane;
      const double *zr = tz + ((kk / 2) * A + jj) * 2 + (kk & 1);
      double next = cf[0];
      for (int s = 0; s < ns; ++s, zr += 4 * A) {
        const double av = next;
        if (s + 1 < ns) next = cf[size_t(s + 1) * kWave];
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = Mfma(av, zr[t * 32], acc[t]);
      }
      const double ny = col.z, nxd = col.y, sy = col.z < 0 ? -1.0 : 1.0;
      if (col.w >= 0) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          double ar, ai;
          if constexpr (XY) {
            const double2 ex = tx[col.y * A + t * 16 + jj], ey = ty[abs(col.z) * A + t * 16 + jj];
            const double eyi = sy * ey.y;
            ar = fma(ex.x, ey.x, -(ex.y * eyi));
            ai = fma(ex.x, eyi, ex.y * ey.x);
          } else {
            const int j = min(a0 + t * 16 + jj, a.natoms - 1);
            const double2 p = PhaseOf(nxd * (a.ux * a.x[j]) + ny * (a.uy * a.y[j]));
            ar = p.x;
            ai = p.y;
          }
          const double f = fma(ar, acc[t][0], ai * acc[t][1]);
          fx[t] = fma(nxd, f, fx[t]);
          fy[t] = fma(ny, f, fy[t]);
          fz[t] = fma(ar, acc[t][2], fma(ai, acc[t][3], fz[t]));
        }
      }
    }
  }
  // the four columns of a lane's atom, then the waves in order
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    double f[3] = {fx[t], fy[t], fz[t]};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      f[d] += __shfl_xor(f[d], 16);
      f[d] += __shfl_xor(f[d], 32);
      if (kk == 0) red[wave][d][t * 16 + jj] = f[d];
    }
  }
  __syncthreads();
  for (int it = tid; it < 3 * A; it += kMmThreads) {
    const int d = it / A, at = it % A, j = a0 + at;
    if (j >= a.natoms) continue;
    double v = 0.0;
    for (int w = 0; w < kMmWaves; ++w) v += red[w][d][at];
    const double q = a.q[j], c = d == 0 ? a.cx : (d == 1 ? a.cy : a.cz);
    a.part[(size_t(chunk) * 3 + d) * a.natoms + j] =
        fabs(q) < 0.000000001 ? 0.0 : (2.0 * q) * (c * v);
  }
}

// Dynamic LDS a kernel may ask for: the 160 KiB of a CU less its static part.
constexpr int kLdsMax = 144 * 1024;

template <int NT, bool XY>
hipError_t LaunchForce(const ForceArgs &a, size_t lds, hipStream_t s) {
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(
        reinterpret_cast<const void *>(&RecipForcePartKernel<NT, XY>),
        hipFuncAttributeMaxDynamicSharedMemorySize, kLdsMax);
    if (e != hipSuccess) return e;
  }
  const int blocks = (a.natoms + 16 * NT - 1) / (16 * NT);
  hipLaunchKernelGGL((RecipForcePartKernel<NT, XY>), dim3(blocks * a.chunks), dim3(kMmThreads), lds, s, a);
  return hipGetLastError();
}

__global__ void ZeroCounterKernel(unsigned *counter) { *counter = 0u; }

}  // namespace

// --------------------------------------------------------------- the plan --
// The box's k-vectors as columns, longest first, and the work units of the
// two products.  Made from the k list whenever it changes.
int BuildKPlan(gomc_box *b, const std::vector<double> &kx, const std::vector<double> &ky,
               const std::vector<double> &kz) {
  KPlan &p = b->kp;
  const int K = int(kx.size());
  double c[3];
  for (int i = 0; i < 3; ++i) c[i] = (1.0 / b->geom.L[i]) * (2.0 * M_PI);  // KVectorsOrth's spacing
  std::vector<int4> cols;
  p.nx = p.ny = p.nz = 0;
  for (int k = 0; k < K;) {
    int e = k + 1;
    while (e < K && kx[e] == kx[k] && ky[e] == ky[k]) ++e;
    const int nx = int(std::rint(kx[k] / c[0])), ny = int(std::rint(ky[k] / c[1])),
              nz = int(std::rint(kz[k] / c[2]));
    const int m = nz + (e - k) - 1;
    if ((nx == 0 && ny == 0) ? nz != 1 : nz != -m)
      return Fail(b, GOMC_ERR_STATE, "k-vectors are not in whole columns of nz");
    cols.push_back(make_int4(k - nz, nx, ny, m));
    p.nx = std::max(p.nx, nx);
    p.ny = std::max(p.ny, std::abs(ny));
    p.nz = std::max(p.nz, m);
    k = e;
  }
  std::stable_sort(cols.begin(), cols.end(), [](const int4 &u, const int4 &v) { return u.w > v.w; });
  const int ncol = int(cols.size());
  while (cols.size() % 16) cols.push_back(make_int4(0, 0, 0, -1));
  // structure factors: (16 columns, 32 nz) units, longest first within a
  // window of nz, dealt to the window's workgroups there and back so that a
  // workgroup's SIMDs (wave w runs on SIMD w % 4) carry alike
  std::vector<int4> dealt;
  for (int w0 = 0; w0 <= p.nz; w0 += 32) {
    std::vector<int4> units;
    for (int g = 0; g < int(cols.size()) / 16; ++g) {
      const int m = cols[size_t(g) * 16].w;
      if (m >= w0) units.push_back(make_int4(g, w0, std::min(4, (m - w0) / 8 + 1), 0));
    }
    const int blocks = int((units.size() + kMmWaves - 1) / kMmWaves);
    for (int g = 0; g < blocks; ++g)
      for (int w = 0; w < kMmWaves; ++w) {
        const size_t u = size_t(w < 4 ? w : 11 - w) * blocks + g;
        dealt.push_back(u < units.size() ? units[u] : make_int4(0, w0, 0, 0));
      }
  }
  p.nB = int(dealt.size() / kMmWaves);
  // forces: groups of 4 columns, two nz a step
  p.ngrp = (ncol + 3) / 4;
  std::vector<int> fstart(1, 0);
  for (int g = 0; g < p.ngrp; ++g) fstart.push_back(fstart.back() + cols[size_t(g) * 4].w / 2 + 1);
  p.steps = fstart.back();
  const size_t nc = cols.size() * 4, nu = dealt.size() * 4, nf = fstart.size();
  std::vector<int> flat(nc + nu + nf);
  std::copy_n(reinterpret_cast<const int *>(cols.data()), nc, flat.begin());
  std::copy_n(reinterpret_cast<const int *>(dealt.data()), nu, flat.begin() + nc);
  std::copy_n(fstart.data(), nf, flat.begin() + nc + nu);
  if (flat.size() > p.cap) {
    if (p.buf) (void)hipFree(p.buf);
    p.buf = nullptr;
    p.cap = 0;
    HIP_TRY(b, hipMalloc(&p.buf, sizeof(int) * flat.size()));
    p.cap = flat.size();
  }
  p.unitOff = nc;
  p.fstartOff = nc + nu;
  HIP_TRY(b, hipMemcpyAsync(p.buf, flat.data(), sizeof(int) * flat.size(), hipMemcpyHostToDevice,
                            b->stream));
  return Sync(b);
}

void FreeKPlan(KPlan &p) {
  for (void *v : {(void *)p.buf, (void *)p.coef})
    if (v) (void)hipFree(v);
  p = KPlan{};
}

// ------------------------------------------------------ structure factors --
constexpr int kSumsTabBytes = 48 * 1024;  // phase tables of a tile
constexpr int kSumsWorkgroups = 512;      // two a CU, what their registers allow

// Atom chunks of the first pass: about kSumsWorkgroups workgroups, chunks of
// at least 32 atoms, chunks x K within kSumsPartCap (pairs of doubles).
static int SumsChunks(const gomc_box *b) {
  int c = (kSumsWorkgroups + b->kp.nB - 1) / std::max(1, b->kp.nB);
  c = std::min(c, (b->natoms + 31) / 32);
  if (b->K > 0) c = std::min<int64_t>(c, int64_t(kSumsPartCap / size_t(b->K)));
  return std::max(1, c);
}

// The box's arrays for the two passes; the scratch (part, partials, counter)
// is the caller's.
static SumsArgs BoxSumsArgs(const gomc_box *b) {
  const KPlan &p = b->kp;
  SumsArgs a;
  a.x = b->x;
  a.y = b->y;
  a.z = b->z;
  a.q = b->q;
  a.mol = b->mol;
  a.natoms = b->natoms;
  a.K = b->K;
  a.cols = reinterpret_cast<const int4 *>(p.buf);
  a.units = reinterpret_cast<const int4 *>(p.buf + p.unitOff);
  a.nB = p.nB;
  a.chunks = SumsChunks(b);
  a.aChunk = (b->natoms + a.chunks - 1) / a.chunks;
  a.Ez = std::min(32, (p.nz + 8) / 8 * 8);
  // a row of 8 mod 16 entries puts four atoms' z reads on different LDS banks
  auto rows = [&](int nx, int ny) {
    a.nx = nx;
    a.ny = ny;
    a.oy = nx + 1;
    a.oz = a.oy + ny + 1;
    a.E = a.oz + a.Ez;
    a.E += (24 - a.E % 16) % 16;
    return size_t(a.E) * sizeof(double2);
  };
  if (4 * rows(p.nx, p.ny) > size_t(kLdsMax)) rows(-1, -1);
  a.T = int(std::max<size_t>(4, std::min<size_t>(64, kSumsTabBytes / (size_t(a.E) * sizeof(double2)) / 4 * 4)));
  a.ux = 2.0 / b->geom.L[0];
  a.uy = 2.0 / b->geom.L[1];
  a.uz = 2.0 / b->geom.L[2];
  a.pref = b->pref;
  a.sumR = b->sumRnew;
  a.sumI = b->sumInew;
  a.result = b->devRes;
  return a;
}

static int SumsBlocks(int K) { return std::max(1, (K + kWave - 1) / kWave); }

static hipError_t LaunchRecipSums(const SumsArgs &a, hipStream_t s) {
  const size_t lds = size_t(a.T) * a.E * sizeof(double2);
  hipError_t e = hipSuccess;
  if (lds > 64 * 1024)
    e = hipFuncSetAttribute(reinterpret_cast<const void *>(&RecipSumsPartKernel<false>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, kLdsMax);
  if (e == hipSuccess && a.nB > 0) {
    const dim3 grid(a.nB * a.chunks);
    if (a.nx < 0)
      hipLaunchKernelGGL(RecipSumsPartKernel<true>, grid, dim3(kMmThreads), lds, s, a);
    else
      hipLaunchKernelGGL(RecipSumsPartKernel<false>, grid, dim3(kMmThreads), lds, s, a);
    e = hipGetLastError();
  }
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(RecipSumsKernel, dim3(SumsBlocks(a.K)), dim3(kBlock), 0, s, a);
  return hipGetLastError();
}

// BoxReciprocalSums into the "new" sums; returns the reciprocal energy.
int RecipSums(gomc_box *b, double *erecip) {
  if (!b->recipReady) return Fail(b, GOMC_ERR_STATE, "k-vectors not initialised");
  SumsArgs a = BoxSumsArgs(b);
  int rc = EnsurePartials(b, SumsBlocks(b->K));
  if (rc) return rc;
  a.partials = b->partials;
  a.counter = b->counter;
  const size_t need = size_t(a.chunks) * size_t(b->K) * 2;
  if (need > b->sumPartCap) {
    if (b->sumPart) (void)hipFree(b->sumPart);
    b->sumPart = nullptr;
    b->sumPartCap = 0;
    HIP_TRY(b, hipMalloc(&b->sumPart, sizeof(double) * need));
    b->sumPartCap = need;
  }
  a.part = reinterpret_cast<double2 *>(b->sumPart);
  HIP_TRY(b, LaunchRecipSums(a, b->stream));
  rc = Sync(b);
  if (rc) return rc;
  *erecip = b->hostRes[2];
  return GOMC_OK;
}

// ------------------------------------------- allocation-free variant --
// gomc_recip_sums_noalloc runs the same two passes as RecipSums with its
// scratch -- the block counter, the second pass's per-block partials and
// the first pass's per-chunk sums -- in `scratch`, one file-scope device
// array that each GPU holds until the process ends.  Layout: counter at
// byte 0, partials at byte 256 (one per 64 k-vectors up to kNoAllocMaxK),
// per-chunk sums after them (SumsChunks keeps chunks x K within
// kSumsPartCap, so 2 kSumsPartCap doubles hold them for K up to
// kNoAllocMaxK).  Every call on one GPU shares the array: calls that
// overlap on one GPU race.
constexpr int kNoAllocMaxK = 1 << 20;
constexpr size_t kNoAllocPartialsOff = 256;
constexpr size_t kNoAllocPartOff =
    kNoAllocPartialsOff + sizeof(Partial4) * size_t(kNoAllocMaxK / kWave);
constexpr size_t kNoAllocPartDoubles = 2 * kSumsPartCap;
constexpr size_t kScratchBytes = kNoAllocPartOff + sizeof(double) * kNoAllocPartDoubles;
static_assert(kNoAllocPartOff % 256 == 0, "per-chunk sums must stay 256-byte aligned");

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kScratchDevices = 64;
static std::mutex gScratchMu;
static unsigned char *gScratch[kScratchDevices] = {};

// Device address of this GPU's `scratch`, looked up once per device with
// that device current (the array's host-side name is not a device address).
static int ScratchBase(gomc_box *b, unsigned char **base) {
  if (b->device < 0 || b->device >= kScratchDevices)
    return Fail(b, GOMC_ERR_ARG, "device index beyond the scratch table");
  std::lock_guard<std::mutex> lock(gScratchMu);
  if (!gScratch[b->device]) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return Fail(b, GOMC_ERR_HIP,
                  std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    gScratch[b->device] = static_cast<unsigned char *>(p);
  }
  *base = gScratch[b->device];
  return GOMC_OK;
}

// The block counter must read zero when the second pass starts; a fill
// kernel, not a memset, so that a captured stream replays it.
int RecipSumsNoAlloc(gomc_box *b, double *erecip) {
  if (!b->recipReady) return Fail(b, GOMC_ERR_STATE, "k-vectors not initialised");
  if (b->K > kNoAllocMaxK)
    return Fail(b, GOMC_ERR_ARG,
                "gomc_recip_sums_noalloc takes at most 1048576 k-vectors (use gomc_recip_sums)");
  SumsArgs a = BoxSumsArgs(b);
  if (size_t(a.chunks) * size_t(b->K) * 2 > kNoAllocPartDoubles)
    return Fail(b, GOMC_ERR_ARG, "structure-factor chunks exceed the scratch array");
  unsigned char *base = nullptr;
  int rc = ScratchBase(b, &base);
  if (rc) return rc;
  a.counter = reinterpret_cast<unsigned *>(base);
  a.partials = reinterpret_cast<Partial4 *>(base + kNoAllocPartialsOff);
  a.part = reinterpret_cast<double2 *>(base + kNoAllocPartOff);
  hipLaunchKernelGGL(ZeroCounterKernel, dim3(1), dim3(1), 0, b->stream, a.counter);
  HIP_TRY(b, hipGetLastError());
  HIP_TRY(b, LaunchRecipSums(a, b->stream));
  rc = Sync(b);
  if (rc) return rc;
  *erecip = b->hostRes[2];
  return GOMC_OK;
}

// ------------------------------------------------------------------ force --
constexpr int kForceWorkgroups = 512;    // two a CU
constexpr int kForceZMax = 32;           // steps of a z window when the tables do not fit
// Tables of a workgroup of 16 nt atoms that leave room for a second one on the
// CU (160 KiB, less the static part).  Measured on cubic water boxes, rc 12 A,
// tolerance 1e-6, microseconds a call with this limit and with 6 KiB more, where
// 64 atoms run alone on a CU instead of 32 and 32 at n = 22 to 24 k-vectors an
// axis: n = 21 113.6 / 113.3, 22 143.0 / 167.2, 23 191.1 / 190.0, 24 215.8 /
// 205.8; 64 atoms alone also at 25 275 / 314, 26 309 / 345, 28 430 / 418, 32 901 /
// 974.
constexpr int ForceTabBytes(int nt) { return 80 * 1024 - int(sizeof(double)) * kMmWaves * 3 * 16 * nt; }

// The k-space force of every atom over the sums (sumR, sumI), as per-chunk
// parts; launched on the box's stream, not waited for.
int RecipForceParts(gomc_box *b, const double *sumR, const double *sumI, RecipParts *out) {
  KPlan &p = b->kp;
  const size_t needC = size_t(std::max(p.steps, 1)) * kWave;
  if (needC > p.coefCap) {
    if (p.coef) (void)hipFree(p.coef);
    p.coef = nullptr;
    p.coefCap = 0;
    HIP_TRY(b, hipMalloc(&p.coef, sizeof(double) * needC));
    p.coefCap = needC;
  }
  CoefArgs c;
  c.cols = reinterpret_cast<const int4 *>(p.buf);
  c.fstart = p.buf + p.fstartOff;
  c.ngrp = p.ngrp;
  c.steps = p.steps;
  c.K = b->K;
  c.pref = b->pref;
  c.sumR = sumR;
  c.sumI = sumI;
  c.coef = p.coef;
  ForceArgs a;
  a.x = b->x;
  a.y = b->y;
  a.z = b->z;
  a.q = b->q;
  a.natoms = b->natoms;
  a.cols = c.cols;
  a.fstart = c.fstart;
  a.ngrp = p.ngrp;
  a.nx = p.nx;
  a.ny = p.ny;
  a.maxSteps = p.nz / 2 + 1;
  a.cx = (1.0 / b->geom.L[0]) * (2.0 * M_PI);
  a.cy = (1.0 / b->geom.L[1]) * (2.0 * M_PI);
  a.cz = (1.0 / b->geom.L[2]) * (2.0 * M_PI);
  a.ux = 2.0 / b->geom.L[0];
  a.uy = 2.0 / b->geom.L[1];
  a.uz = 2.0 / b->geom.L[2];
  a.coef = p.coef;
  // atoms per workgroup: 64, halved while the tables leave no room for a
  // second workgroup on the CU (a long box); beyond 16, z in windows and, if
  // x and y alone are too long, no tables for them
  bool xy = true;
  a.zSteps = a.maxSteps;
  auto bytes = [&](int A) {
    return (xy ? size_t(a.nx + a.ny + 2) * A * sizeof(double2) : 0) +
           size_t(4) * a.zSteps * A * sizeof(double);
  };
  int nt = 4;
  while (nt > 1 && bytes(16 * nt) > size_t(ForceTabBytes(nt))) nt /= 2;
  if (bytes(16 * nt) > size_t(ForceTabBytes(nt))) a.zSteps = std::min(a.zSteps, kForceZMax);
  if (bytes(16 * nt) > size_t(ForceTabBytes(nt))) xy = false;
  const int blocks = (b->natoms + 16 * nt - 1) / (16 * nt);
  const int most = std::max(1, (p.ngrp + kMmWaves - 1) / kMmWaves);
  a.chunks = std::max(1, std::min(most, (kForceWorkgroups + blocks / 2) / std::max(1, blocks)));
  const size_t need = size_t(a.chunks) * 3 * size_t(std::max(b->natoms, 1));
  if (need > b->forcePartCap) {
    if (b->forcePart) (void)hipFree(b->forcePart);
    b->forcePart = nullptr;
    b->forcePartCap = 0;
    HIP_TRY(b, hipMalloc(&b->forcePart, sizeof(double) * need));
    b->forcePartCap = need;
  }
  a.part = b->forcePart;
  if (p.steps > 0) {
    const int per = kBlock / kWave;
    hipLaunchKernelGGL(RecipCoefKernel, dim3((p.steps + per - 1) / per), dim3(kBlock), 0, b->stream,
                       c);
    HIP_TRY(b, hipGetLastError());
  }
  const size_t lds = bytes(16 * nt);
  const hipError_t e = !xy       ? LaunchForce<1, false>(a, lds, b->stream)
                       : nt == 4 ? LaunchForce<4, true>(a, lds, b->stream)
                       : nt == 2 ? LaunchForce<2, true>(a, lds, b->stream)
                                 : LaunchForce<1, true>(a, lds, b->stream);
  HIP_TRY(b, e);
  out->part = a.part;
  out->chunks = a.chunks;
  return GOMC_OK;
}

}  // namespace gomc
