// Molecular virial and pressure of a box (CalculateEnergy::VirialCalc,
// src/CalculateEnergy.cpp:411-579; VirialCorrection 1317-1336;
// Ewald::VirialReciprocal, src/Ewald.cpp:1168-1305; the pressure of
// OutputVars.cpp:147-172), diagonal tensor terms as in the reference.
//
// The pair part comes per block from pair.hip and the k-space forces from
// recip.hip; RecipVirialKernel makes the reciprocal part per block, and
// VirialSumKernel adds all blocks.
#include <algorithm>
#include <cmath>

#include "box.hpp"

namespace {
using namespace gomc;

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
    if (threadIdx.x == 0) a.part[size_t(blockIdx.x) * 3 + c] = s;
  }
}

// result = {LJ xx yy zz, real xx yy zz, reciprocal xx yy zz}: one wave per
// component, a lane the blocks lane, lane + 64, ... in order.
struct VirialSumArgs {
  const double *pair, *recip;
  int npair, nrecip;
  double *result;
};

__global__ void __launch_bounds__(9 * kWave) VirialSumKernel(const VirialSumArgs a) {
  const int lane = threadIdx.x % kWave, c = threadIdx.x / kWave;
  const double *p = c < 6 ? a.pair + c : a.recip + (c - 6);
  const int n = c < 6 ? a.npair : a.nrecip, stride = c < 6 ? 6 : 3;
  double s = 0.0;
#pragma unroll 8
  for (int i = lane; i < n; i += kWave) s += p[size_t(i) * stride];
  s = WaveSum(s);
  if (lane == 0) a.result[c] = s;
}

}  // namespace

extern "C" int gomc_box_virial(gomc_box *b, double out[9]) {
  if (!b || !out) return GOMC_ERR_ARG;
  (void)hipSetDevice(b->device);
  int rc = FlushPending(b);
  if (!rc) rc = MPEnsure(b);
  if (!rc) rc = MPUploadCom(b);  // molecule centres of the current coordinates
  VirialSumArgs v;
  if (!rc) rc = PairVirials(b, b->mp.com[0], &v.pair, &v.npair);
  if (rc) return rc;
  const int kBlocks = b->ewald ? (b->K + kBlock - 1) / kBlock : 0;
  const int atomBlocks = b->ewald ? (b->natoms + kBlock - 1) / kBlock : 0;
  const size_t need = size_t(3) * (kBlocks + atomBlocks);
  if (need > b->virCap) {  // grows only with the box's block count
    if (b->virBuf) (void)hipFree(b->virBuf);
    b->virBuf = nullptr;
    b->virCap = 0;
    HIP_TRY(b, hipMalloc(&b->virBuf, sizeof(double) * need));
    b->virCap = need;
  }
  if (b->ewald) {
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
    r.cx = b->mp.com[0][0];
    r.cy = b->mp.com[0][1];
    r.cz = b->mp.com[0][2];
    r.constVal = 1.0 / (4.0 * (b->alpha * b->alpha));
    r.part = b->virBuf;
    hipLaunchKernelGGL(RecipVirialKernel, dim3(kBlocks + atomBlocks), dim3(kBlock), 0, b->stream, r);
    HIP_TRY(b, hipGetLastError());
  }
  v.recip = b->virBuf;
  v.nrecip = kBlocks + atomBlocks;
  v.result = b->devRes;
  hipLaunchKernelGGL(VirialSumKernel, dim3(1), dim3(9 * kWave), 0, b->stream, v);
  HIP_TRY(b, hipGetLastError());
  rc = Sync(b);
  if (rc) return rc;
  const double *vT = b->hostRes, *rT = b->hostRes + 3, *wT = b->hostRes + 6;
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
