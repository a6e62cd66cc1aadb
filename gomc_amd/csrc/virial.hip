// Molecular virial and pressure of a box (CalculateEnergy::VirialCalc,
// src/CalculateEnergy.cpp:411-579; VirialCorrection 1317-1336;
// Ewald::VirialReciprocal, src/Ewald.cpp:1168-1305; the pressure of
// OutputVars.cpp:147-172), diagonal tensor terms as in the reference.
//
// PairVirialKernel: one workgroup per (cell, neighbour slot), the same
// enumeration as BoxInterKernel: for every inter-molecular pair inside the
// box cutoff, F/r of the LJ and erfc-Coulomb terms times the atom
// separation's and the minimum-image centre separation's components.  A
// wave takes (64 cell atoms, 64 neighbour atoms) items and queues their
// in-cutoff pairs in its LDS, so the pair terms run once per 64 queued
// pairs, not once per 64 tested.
// RecipVirialKernel: the reciprocal part.  Each block writes its partial
// sums; the host adds them in block order.
#include <algorithm>
#include <cmath>

#include "box.hpp"

namespace {
using namespace gomc;

constexpr int kVirSlots = 8;

struct PairVirArgs {
  BoxGeom g;
  const double *x, *y, *z, *q;
  const int *type, *mol;
  const double *sigSq, *epsCn6, *nOver6, *nHalf;
  int ntypes;
  const int *cellStart, *cellVec, *nbr;
  const double *cx, *cy, *cz;  // molecule centres
  double *part;                // [blocks][kVirSlots]
};

constexpr int kUnroll = 4;  // neighbour entries tested per step of the pair virial

// 64 atoms of a cell staged in a wave's LDS, with their molecules' centres.
struct VirTile {
  double x[kWave], y[kWave], z[kWave], q[kWave], cx[kWave], cy[kWave], cz[kWave];
  int idx[kWave], type[kWave], mol[kWave];
};

__device__ __forceinline__ void StageVirTile(const PairVirArgs &a, VirTile &t, int first, int n,
                                             int lane) {
  if (lane < n) {
    const int j = a.cellVec[first + lane], m = a.mol[j];
    t.idx[lane] = j;
    t.x[lane] = a.x[j];
    t.y[lane] = a.y[j];
    t.z[lane] = a.z[j];
    t.q[lane] = a.q[j];
    t.type[lane] = a.type[j];
    t.mol[lane] = m;
    t.cx[lane] = a.cx[m];
    t.cy[lane] = a.cy[m];
    t.cz[lane] = a.cz[m];
  }
}

// The virial terms of one in-cutoff pair (entry u of tile I, entry k of
// tile J) added to v: FFParticle::CalcCoulombVir and CalcVir
// (FFParticle.cpp:295-359, 401-446) times the atom and centre separations'
// components, the Coulomb term with erfc(a r) = exp(-(a r)^2) erfcx(a r)
// where the reference writes 1 - erf.
__device__ __forceinline__ void PairVirial(const PairVirArgs &a, const double *poly,
                                           const VirTile &I, int u, const VirTile &J, int k,
                                           double v[6]) {
  const double dx = MinImage(I.x[u] - J.x[k], a.g.L[0], a.g.half[0]);
  const double dy = MinImage(I.y[u] - J.y[k], a.g.L[1], a.g.half[1]);
  const double dz = MinImage(I.z[u] - J.z[k], a.g.L[2], a.g.half[2]);
  const double d2 = dx * dx + dy * dy + dz * dz;
  const double cdx = MinImage(I.cx[u] - J.cx[k], a.g.L[0], a.g.half[0]);
  const double cdy = MinImage(I.cy[u] - J.cy[k], a.g.L[1], a.g.half[1]);
  const double cdz = MinImage(I.cz[u] - J.cz[k], a.g.L[2], a.g.half[2]);
  const int idx = I.type[u] + J.type[k] * a.ntypes;
  const PairTerms t = PairMath(a.g, poly, d2, I.q[u] * J.q[k], a.sigSq[idx], 0.0, a.nHalf[idx],
                               a.epsCn6[idx], a.nOver6[idx], false);
  v[0] += t.vLJ * (dx * cdx);
  v[1] += t.vLJ * (dy * cdy);
  v[2] += t.vLJ * (dz * cdz);
  v[3] += t.vReal * (dx * cdx);
  v[4] += t.vReal * (dy * cdy);
  v[5] += t.vReal * (dz * cdz);
}

__device__ __forceinline__ void WaveSync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The block's (cell chunk of 64, neighbour tile of 64) items go to its
// waves round robin.  A wave stages both tiles in its LDS, each lane holds
// one cell atom and walks the neighbour tile kUnroll entries at a time, and
// the in-cutoff pairs are queued; the pair terms run once per 64 queued
// pairs (and once for an item's rest).  The sums' order is fixed by the
// positions.
__global__ void __launch_bounds__(kBlock, 4) PairVirialKernel(const PairVirArgs a) {
  constexpr int kWaves = kBlock / kWave;
  __shared__ VirTile tileI[kWaves], tileJ[kWaves];
  __shared__ int pairList[kWaves][(kUnroll + 1) * kWave];
  __shared__ double red[kWaves];
  __shared__ double poly[kErfcxDeg + 1];
  if (threadIdx.x <= kErfcxDeg) poly[threadIdx.x] = kErfcxPoly[threadIdx.x];
  __syncthreads();
  const int cell = blockIdx.x / 27, nb = a.nbr[blockIdx.x];
  const int cs = a.cellStart[cell], ce = a.cellStart[cell + 1];
  const int ns = a.cellStart[nb], ne = a.cellStart[nb + 1];
  const int ic = (ce - cs + kWave - 1) / kWave, jc = (ne - ns + kWave - 1) / kWave;
  const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
  VirTile &I = tileI[w], &J = tileJ[w];
  int *q = pairList[w];
  const uint64_t below = (uint64_t(1) << lane) - 1;
  double v[6] = {0, 0, 0, 0, 0, 0};  // LJ xx yy zz, real xx yy zz
  for (int item = w; item < ic * jc; item += kWaves) {
    const int i0 = cs + (item / jc) * kWave, j0 = ns + (item % jc) * kWave;
    const int ni = min(kWave, ce - i0), nj = min(kWave, ne - j0);
    WaveSync();  // the previous item's reads are done
    StageVirTile(a, I, i0, ni, lane);
    StageVirTile(a, J, j0, nj, lane);
    WaveSync();
    const bool iv = lane < ni;
    const int i = iv ? I.idx[lane] : 0, mi = iv ? I.mol[lane] : -1;
    const double xi = iv ? I.x[lane] : 0.0, yi = iv ? I.y[lane] : 0.0, zi = iv ? I.z[lane] : 0.0;
    // kUnroll tile entries per step, each lane testing its atom against
    // them; the wave queues the in-cutoff pairs (i < j, other molecule)
    int queued = 0;
    for (int k0 = 0; k0 < nj || queued > 0; k0 += kUnroll) {
      if (k0 < nj) {
        bool hit[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
          const int k = k0 + u;
          hit[u] = false;
          if (iv && k < nj && i < J.idx[k] && mi != J.mol[k]) {
            const double dx = MinImage(xi - J.x[k], a.g.L[0], a.g.half[0]);
            const double dy = MinImage(yi - J.y[k], a.g.L[1], a.g.half[1]);
            const double dz = MinImage(zi - J.z[k], a.g.L[2], a.g.half[2]);
            hit[u] = a.g.rCutSq > dx * dx + dy * dy + dz * dz;
          }
        }
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
          const uint64_t m = __ballot(hit[u]);
          if (hit[u]) q[queued + __popcll(m & below)] = (lane << 6) | (k0 + u);
          queued += __popcll(m);
        }
      }
      // full batches, or the item's last pairs
      while (queued >= kWave || (queued > 0 && k0 + kUnroll >= nj)) {
        WaveSync();
        const int n = min(queued, kWave);
        if (lane < n) {
          const int e = q[queued - n + lane];
          PairVirial(a, poly, I, e >> 6, J, e & 63, v);
        }
        queued -= n;
        WaveSync();
      }
    }
  }
  for (int c = 0; c < 6; ++c) {
    const double s = BlockSum(v[c], red);
    if (threadIdx.x == 0) a.part[size_t(blockIdx.x) * kVirSlots + c] = s;
  }
}

// The reciprocal part: blocks [0, kBlocks) one k-vector per thread (the
// k-space term); the others one atom per thread (the intramolecular term:
// minus the atom's k-space force, in parts from recip.hip's matrix product,
// times its offset from its molecule's centre).
struct RecipVirArgs {
  BoxGeom g;
  const double *x, *y, *z, *q;
  const int *mol;
  int natoms, K, kBlocks;
  RecipParts f;
  const double *kx, *ky, *kz, *pref, *sumR, *sumI;
  const double *cx, *cy, *cz;
  double constVal;  // 1 / (4 alpha^2)
  double *part;
};

__global__ void __launch_bounds__(kBlock) RecipVirialKernel(const RecipVirArgs a) {
  __shared__ double red[kBlock / kWave];
  double w[3] = {0, 0, 0};
  if (int(blockIdx.x) < a.kBlocks) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i < a.K) {
      const double kx = a.kx[i], ky = a.ky[i], kz = a.kz[i];
      const double hsqr = kx * kx + ky * ky + kz * kz;
      const double factor = a.pref[i] * (a.sumR[i] * a.sumR[i] + a.sumI[i] * a.sumI[i]);
      w[0] = factor * (1.0 - 2.0 * (a.constVal + 1.0 / hsqr) * kx * kx);
      w[1] = factor * (1.0 - 2.0 * (a.constVal + 1.0 / hsqr) * ky * ky);
      w[2] = factor * (1.0 - 2.0 * (a.constVal + 1.0 / hsqr) * kz * kz);
    }
  } else {
    const int p = (blockIdx.x - a.kBlocks) * kBlock + threadIdx.x;
    const int m = p < a.natoms ? a.mol[p] : -1;
    if (m >= 0 && !(fabs(a.q[p]) < 0.000000001)) {
      const double r[3] = {a.x[p], a.y[p], a.z[p]}, c[3] = {a.cx[m], a.cy[m], a.cz[m]};
      double f[3] = {0, 0, 0};
#pragma unroll 4
      for (int ch = 0; ch < a.f.chunks; ++ch) {
        const double *part = a.f.part + size_t(ch) * 3 * a.natoms + p;
        f[0] += part[0];
        f[1] += part[a.natoms];
        f[2] += part[2 * size_t(a.natoms)];
      }
#pragma unroll
      for (int d = 0; d < 3; ++d)
        w[d] = -f[d] * (Unwrap(r[d], c[d], a.g.L[d], a.g.half[d]) - c[d]);
    }
  }
  for (int c = 0; c < 3; ++c) {
    const double s = BlockSum(w[c], red);
    if (threadIdx.x == 0) a.part[size_t(blockIdx.x) * kVirSlots + c] = s;
  }
}

}  // namespace

extern "C" int gomc_box_virial(gomc_box *b, double out[9]) {
  if (!b || !out) return GOMC_ERR_ARG;
  (void)hipSetDevice(b->device);
  int rc = FlushPending(b);
  if (!rc) rc = MPEnsure(b);
  if (!rc) rc = MPUploadCom(b);  // molecule centres of the current coordinates
  if (!rc) rc = BuildCells(b);
  if (rc) return rc;
  const int pairBlocks = b->ncell * 27;
  const int kBlocks = b->ewald ? (b->K + kBlock - 1) / kBlock : 0;
  const int atomBlocks = b->ewald ? (b->natoms + kBlock - 1) / kBlock : 0;
  const int nblocks = pairBlocks + kBlocks + atomBlocks;
  const size_t need = size_t(kVirSlots) * std::max(nblocks, 1);
  if (need > b->virCap) {  // grows only with the box's block count
    if (b->virBuf) (void)hipFree(b->virBuf);
    b->virBuf = nullptr;
    b->virCap = 0;
    HIP_TRY(b, hipMalloc(&b->virBuf, sizeof(double) * need));
    b->virCap = need;
  }
  double *part = b->virBuf;
  PairVirArgs a;
  a.g = b->geom;
  a.x = b->x;
  a.y = b->y;
  a.z = b->z;
  a.q = b->q;
  a.type = b->type;
  a.mol = b->mol;
  a.sigSq = b->tSigSq;
  a.epsCn6 = b->tEpsCn6;
  a.nOver6 = b->tNOver6;
  a.nHalf = b->tNHalf;
  a.ntypes = b->ntypes;
  a.cellStart = b->cellStart;
  a.cellVec = b->cellVec;
  a.nbr = b->nbr;
  a.cx = b->mp.com[0][0];
  a.cy = b->mp.com[0][1];
  a.cz = b->mp.com[0][2];
  a.part = part;
  hipLaunchKernelGGL(PairVirialKernel, dim3(pairBlocks), dim3(kBlock), 0, b->stream, a);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess && b->ewald) {
    RecipVirArgs r;
    rc = RecipForceParts(b, b->sumRref, b->sumIref, &r.f);
    if (rc) return rc;
    r.g = b->geom;
    r.x = b->x;
    r.y = b->y;
    r.z = b->z;
    r.q = b->q;
    r.mol = b->mol;
    r.natoms = b->natoms;
    r.K = b->K;
    r.kBlocks = kBlocks;
    r.kx = b->kx;
    r.ky = b->ky;
    r.kz = b->kz;
    r.pref = b->pref;
    r.sumR = b->sumRref;
    r.sumI = b->sumIref;
    r.cx = a.cx;
    r.cy = a.cy;
    r.cz = a.cz;
    r.constVal = 1.0 / (4.0 * (b->alpha * b->alpha));
    r.part = part + size_t(pairBlocks) * kVirSlots;
    hipLaunchKernelGGL(RecipVirialKernel, dim3(kBlocks + atomBlocks), dim3(kBlock), 0,
                       b->stream, r);
    e = hipGetLastError();
  }
  std::vector<double> h(size_t(kVirSlots) * std::max(nblocks, 1), 0.0);
  if (e == hipSuccess)
    e = hipMemcpyAsync(h.data(), part, sizeof(double) * kVirSlots * nblocks, hipMemcpyDeviceToHost,
                       b->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(b->stream);
  if (e != hipSuccess) return HipFail(b, e, "virial kernels");
  double vT[3] = {0, 0, 0}, rT[3] = {0, 0, 0}, wT[3] = {0, 0, 0};
  for (int blk = 0; blk < pairBlocks; ++blk)
    for (int d = 0; d < 3; ++d) {
      vT[d] += h[size_t(blk) * kVirSlots + d];
      rT[d] += h[size_t(blk) * kVirSlots + 3 + d];
    }
  for (int blk = pairBlocks; blk < nblocks; ++blk)
    for (int d = 0; d < 3; ++d) wT[d] += h[size_t(blk) * kVirSlots + d];
  const double inter = vT[0] + vT[1] + vT[2];
  const double real = b->elect ? (rT[0] + rT[1] + rT[2]) * kQQFact : 0.0;
  double tail = 0.0;  // VirialCorrection
  if (b->lrc)
    for (int i = 0; i < b->nkinds; ++i)
      for (int j = 0; j < b->nkinds; ++j)
        tail += b->pairVirCorr[i * b->nkinds + j] * unsigned(b->kindCount[i]) *
                unsigned(b->kindCount[j]) * b->volInv;
  const double recip = wT[0] + wT[1] + wT[2];
  out[0] = inter;
  out[1] = tail;
  out[2] = real;
  out[3] = recip;
  out[4] = inter + tail + real + recip;
  // the pressure: each term over the dimensionality and the volume, the
  // ideal part from the number densities, K molecule / A^3 to bar
  const double V = b->volume;
  const double total = inter / 3.0 / V + tail / 3.0 / V + real / 3.0 / V + recip / 3.0 / V;
  double raw = 0.0;
  for (int k = 0; k < b->nkinds; ++k) raw += b->kindCount[k] * b->volInv;
  raw *= b->T;
  raw += total;
  out[5] = raw * 138.0649;
  for (int d = 0; d < 3; ++d) out[6 + d] = vT[d] + (b->elect ? rT[d] * kQQFact : 0.0) + wT[d];
  return GOMC_OK;
}
