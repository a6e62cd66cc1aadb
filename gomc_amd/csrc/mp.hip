// MultiParticle move on the plain path (src/moves/MultiParticle.h): the
// pair forces of CalculateEnergy::BoxForce, the reciprocal forces of
// Ewald::BoxForceReciprocal, molecule forces and torques
// (CalculateEnergy::CalculateTorque), the force-biased transform of every
// molecule (MultiParticle::CalculateTrialDistRot) and the acceptance
// coefficient (MultiParticle::GetCoeff), all on device-resident state.
//
// Forces are summed per atom over the full neighbourhood (each pair is
// evaluated from both ends) instead of scattered with atomics, so every
// sum has a fixed order and a run is reproducible bit for bit.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "box.hpp"

using namespace gomc;

namespace {

constexpr double kMinForce = 1E-12, kMaxForce = 30;  // MultiParticle.h:18-19
constexpr double kLambda = 0.5;                      // MultiParticle.h:95

struct Vec3D {
  double x, y, z;
};

// r123::uneg11<double> for a 64-bit word (lib/Random123/uniform.hpp:196-214).
__device__ __forceinline__ double Uneg11(uint64_t v) {
  return double(int64_t(v)) * 0x1p-63 + 0x1p-64;
}

// ------------------------------------------------------ reciprocal force --
// Ewald::BoxForceReciprocal (Ewald.cpp:1496-1596): the k-space force of
// every atom comes in parts from the matrix product of recip.hip; here, one
// atom per thread, the intramolecular erf correction is subtracted and the
// parts are added in order.
struct RecipForceArgs {
  BoxGeom g;
  const double *x, *y, *z, *q;
  const int *mol, *molStart;
  int natoms;
  double *fx, *fy, *fz;
  RecipParts k;
};

__global__ void __launch_bounds__(kWave) RecipForceKernel(const RecipForceArgs a) {
  const int p = blockIdx.x * kWave + threadIdx.x;
  if (p >= a.natoms) return;
  double X = 0.0, Y = 0.0, Z = 0.0;
  const double xp = a.x[p], yp = a.y[p], zp = a.z[p], qp = a.q[p];
  if (!(fabs(qp) < 0.000000001)) {
    const int m = a.mol[p];  // < 0: a reservoir atom, no intramolecular term
    const int s = m < 0 ? p : a.molStart[m], e = m < 0 ? p : a.molStart[m + 1];
    const double constValue = a.g.alpha * M_2_SQRTPI;
    const double alphaSq = a.g.alpha * a.g.alpha;
    for (int j = s; j < e; ++j) {
      if (j == p) continue;
      const double dx = MinImage(xp - a.x[j], a.g.L[0], a.g.half[0]);
      const double dy = MinImage(yp - a.y[j], a.g.L[1], a.g.half[1]);
      const double dz = MinImage(zp - a.z[j], a.g.L[2], a.g.half[2]);
      const double distSq = dx * dx + dy * dy + dz * dz;
      const double dist = sqrt(distSq);
      const double expConstValue = exp(-1.0 * alphaSq * distSq);
      const double qiqj = qp * a.q[j] * kQQFact;
      double intraForce = qiqj * 1.0 * 1.0 / distSq;
      intraForce *= ((erf(a.g.alpha * dist) / dist) - constValue * expConstValue);
      X -= intraForce * dx;
      Y -= intraForce * dy;
      Z -= intraForce * dz;
    }
  }
#pragma unroll 4
  for (int c = 0; c < a.k.chunks; ++c) {
    const double *part = a.k.part + size_t(c) * 3 * a.natoms + p;
    X += part[0];
    Y += part[a.natoms];
    Z += part[2 * size_t(a.natoms)];
  }
  a.fx[p] = X;
  a.fy[p] = Y;
  a.fz[p] = Z;
}

// ------------------------------------------------ molecule terms, torque --
// One molecule per thread: the molecule sums of the atom forces (the
// reference accumulates them pair by pair, CalculateEnergy.cpp:373-378,
// and atom by atom, Ewald.cpp:1586) and the torque about the molecule's
// centre (CalculateEnergy.cpp:1384-1398).  `mode` bit 0: pair sums,
// bit 1: reciprocal sums, bit 2: torque.
struct MolTermsArgs {
  BoxGeom g;
  const double *x, *y, *z, *cx, *cy, *cz;
  const int *molStart;
  int nmols, mode;
  const double *aF[3], *aFR[3];
  double *mF[3], *mFR[3], *tq[3];
};

__global__ void __launch_bounds__(kBlock) MolTermsKernel(const MolTermsArgs a) {
  const int m = blockIdx.x * kBlock + threadIdx.x;
  if (m >= a.nmols) return;
  const int s = a.molStart[m], e = a.molStart[m + 1];
  if (a.mode & 1)
    for (int d = 0; d < 3; ++d) {
      double v = 0.0;
      for (int p = s; p < e; ++p) v += a.aF[d][p];
      a.mF[d][m] = v;
    }
  if (a.mode & 2)
    for (int d = 0; d < 3; ++d) {
      double v = 0.0;
      for (int p = s; p < e; ++p) v += a.aFR[d][p];
      a.mFR[d][m] = v;
    }
  if (a.mode & 4) {
    const double c[3] = {a.cx[m], a.cy[m], a.cz[m]};
    double tx = 0.0, ty = 0.0, tz = 0.0;
    for (int p = s; p < e; ++p) {
      const double dx = MinImage(a.x[p] - c[0], a.g.L[0], a.g.half[0]);
      const double dy = MinImage(a.y[p] - c[1], a.g.L[1], a.g.half[1]);
      const double dz = MinImage(a.z[p] - c[2], a.g.L[2], a.g.half[2]);
      const double fx = a.aF[0][p] + a.aFR[0][p], fy = a.aF[1][p] + a.aFR[1][p],
                   fz = a.aF[2][p] + a.aFR[2][p];
      tx += dy * fz - dz * fy;
      ty += dz * fx - dx * fz;
      tz += dx * fy - dy * fx;
    }
    a.tq[0][m] = tx;
    a.tq[1][m] = ty;
    a.tq[2][m] = tz;
  }
}

// ------------------------------------------------------------- transform --
// MultiParticle::CalculateTrialDistRot (MultiParticle.h:565-611) with
// CalcRandomTransform (546-563), Rotate/TranslateForceBiased (613-665) and
// Rotate/TranslateRandom (667-712): one molecule per thread, Philox4x64-10
// with key {step, seed} and counter {molecule, 0, 0, 0}
// (Random123Wrapper.cpp:16-22).  A displacement beyond half the box in any
// component, or a non-finite transform, sets `fail` (MultiParticle.h:366-406).
struct TransformArgs {
  BoxGeom g;
  int nmols, rotate;
  uint64_t step, seed;
  double beta, max;
  const double *x, *y, *z, *cx, *cy, *cz;
  double *xn, *yn, *zn, *ncx, *ncy, *ncz;
  const int *molStart;
  const double *mF[3], *mFR[3], *tq[3];
  double *tk[3];
  int *inRange;
  double *fail;  // host-mapped
};

// TransformMatrix::FromAxisAngle (src/TransformMatrix.h:186-214).
__device__ void AxisAngleDev(double theta, const double ax[3], double r[3][3]) {
  const double cross[3][3] = {{0.0, -ax[2], ax[1]}, {ax[2], 0.0, -ax[0]}, {-ax[1], ax[0], 0.0}};
  const double c = cos(theta), s = sin(theta);
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j) {
      const double tensor = ax[i] * ax[j];
      r[i][j] = (i == j ? c : 0.0) + (s * cross[i][j] + (1 - c) * tensor);
    }
}

__global__ void __launch_bounds__(kBlock) TransformKernel(const TransformArgs a) {
  const int m = blockIdx.x * kBlock + threadIdx.x;
  if (m >= a.nmols) return;
  double lb[3], lbmax[3];
  for (int d = 0; d < 3; ++d) {
    lb[d] = a.rotate ? (a.tq[d][m] * kLambda) * a.beta : ((a.mF[d][m] + a.mFR[d][m]) * kLambda) * a.beta;
    lbmax[d] = lb[d] * a.max;
  }
  bool in = true;
  for (int d = 0; d < 3; ++d) in = in && fabs(lbmax[d]) > kMinForce && fabs(lbmax[d]) < kMaxForce;
  const U64x4 r = Philox(uint64_t(uint32_t(m)), 0, 0, 0, a.step, a.seed);
  double val[3] = {0.0, 0.0, 0.0};
  if (in)
    for (int d = 0; d < 3; ++d)
      val[d] = log(exp(-1.0 * lbmax[d]) + 2.0 * U01(r.v[d]) * sinh(lbmax[d])) / lb[d];
  for (int d = 0; d < 3; ++d) a.tk[d][m] = val[d];
  a.inRange[m] = in ? 1 : 0;
  bool bad = !isfinite(sqrt(val[0] * val[0] + val[1] * val[1] + val[2] * val[2]));
  if (!a.rotate && (val[0] > a.g.half[0] || val[1] > a.g.half[1] || val[2] > a.g.half[2])) bad = true;
  if (bad) *a.fail = 1.0;

  const int s = a.molStart[m], e = a.molStart[m + 1];
  const double c[3] = {a.cx[m], a.cy[m], a.cz[m]};
  if (!a.rotate) {
    double sh[3];
    for (int d = 0; d < 3; ++d) sh[d] = in ? val[d] : a.max * Uneg11(r.v[d]);
    for (int p = s; p < e; ++p) {
      a.xn[p] = Wrap(a.x[p] + sh[0], a.g.L[0]);
      a.yn[p] = Wrap(a.y[p] + sh[1], a.g.L[1]);
      a.zn[p] = Wrap(a.z[p] + sh[2], a.g.L[2]);
    }
    a.ncx[m] = Wrap(c[0] + sh[0], a.g.L[0]);
    a.ncy[m] = Wrap(c[1] + sh[1], a.g.L[1]);
    a.ncz[m] = Wrap(c[2] + sh[2], a.g.L[2]);
    return;
  }
  double theta, ax[3];
  if (in) {
    theta = sqrt(val[0] * val[0] + val[1] * val[1] + val[2] * val[2]);
    const double inv = 1.0 / theta;
    for (int d = 0; d < 3; ++d) ax[d] = val[d] * inv;
  } else {
    theta = a.max * Uneg11(r.v[0]);
    const double u = Uneg11(r.v[1]);
    const double th = 2.0 * M_PI * U01(r.v[2]);
    const double root = sqrt(1.0 - u * u);
    ax[0] = root * cos(th);
    ax[1] = root * sin(th);
    ax[2] = u;
  }
  double R[3][3];
  AxisAngleDev(theta, ax, R);
  for (int p = s; p < e; ++p) {
    double v[3] = {Unwrap(a.x[p], c[0], a.g.L[0], a.g.half[0]) + (-c[0]),
                   Unwrap(a.y[p], c[1], a.g.L[1], a.g.half[1]) + (-c[1]),
                   Unwrap(a.z[p], c[2], a.g.L[2], a.g.half[2]) + (-c[2])};
    double w[3];
    for (int i = 0; i < 3; ++i) w[i] = R[i][0] * v[0] + R[i][1] * v[1] + R[i][2] * v[2];
    a.xn[p] = Wrap(w[0] + c[0], a.g.L[0]);
    a.yn[p] = Wrap(w[1] + c[1], a.g.L[1]);
    a.zn[p] = Wrap(w[2] + c[2], a.g.L[2]);
  }
  a.ncx[m] = c[0];
  a.ncy[m] = c[1];
  a.ncz[m] = c[2];
}

// ----------------------------------------------------------- coefficient --
// MultiParticle::GetCoeff / CalculateWRatio (MultiParticle.h:445-511): the
// product over in-range molecules of the forward/backward weight ratios,
// a fixed tree within each workgroup, then workgroups in index order.
struct CoeffArgs {
  int nmols, rotate;
  double lBeta, max;
  const double *tk[3];
  const int *inRange;
  const double *nF[3], *nFR[3], *nT[3], *oF[3], *oFR[3], *oT[3];
  double *parts;
  unsigned *counter;
  double *result;
};

__device__ double WRatio(const double n[3], const double o[3], const double k[3], double max) {
  double w = 1.0;
  for (int d = 0; d < 3; ++d) {
    w *= n[d] * exp(-n[d] * k[d]) / (2.0 * sinh(n[d] * max));
    w /= o[d] * exp(o[d] * k[d]) / (2.0 * sinh(o[d] * max));
  }
  return w;
}

__global__ void __launch_bounds__(kBlock) CoeffKernel(const CoeffArgs a) {
  __shared__ double sw[kBlock];
  __shared__ bool last;
  const int m = blockIdx.x * kBlock + threadIdx.x;
  double w = 1.0;
  if (m < a.nmols && a.inRange[m]) {
    double n[3], o[3], k[3];
    for (int d = 0; d < 3; ++d) {
      k[d] = a.tk[d][m];
      if (a.rotate) {
        n[d] = a.nT[d][m] * a.lBeta;
        o[d] = a.oT[d][m] * a.lBeta;
      } else {
        n[d] = (a.nF[d][m] + a.nFR[d][m]) * a.lBeta;
        o[d] = (a.oF[d][m] + a.oFR[d][m]) * a.lBeta;
      }
    }
    w = WRatio(n, o, k, a.max);
  }
  sw[threadIdx.x] = w;
  __syncthreads();
  for (int s = kBlock / 2; s > 0; s >>= 1) {
    if (int(threadIdx.x) < s) sw[threadIdx.x] *= sw[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    a.parts[blockIdx.x] = sw[0];
    __threadfence();
    last = (atomicAdd(a.counter, 1u) == gridDim.x - 1);
  }
  __syncthreads();
  if (last && threadIdx.x == 0) {
    __threadfence();
    volatile double *vp = a.parts;
    double p = 1.0;
    for (unsigned i = 0; i < gridDim.x; ++i) p *= vp[i];
    *a.result = p;
    *a.counter = 0u;
    __threadfence_system();
  }
}

}  // namespace

namespace gomc {

void MPFree(gomc_box *b) {
  MPState &mp = b->mp;
  std::vector<void *> ptrs = {mp.xn, mp.yn, mp.zn, mp.inRange, mp.wpart,
                              mp.wcounter};
  for (int s = 0; s < 2; ++s)
    for (int d = 0; d < 3; ++d) {
      ptrs.push_back(mp.com[s][d]);
      ptrs.push_back(mp.aF[s][d]);
      ptrs.push_back(mp.aFR[s][d]);
      ptrs.push_back(mp.mF[s][d]);
      ptrs.push_back(mp.mFR[s][d]);
      ptrs.push_back(mp.tq[s][d]);
    }
  for (int d = 0; d < 3; ++d) ptrs.push_back(mp.tk[d]);
  for (void *p : ptrs)
    if (p) (void)hipFree(p);
  mp = MPState{};
}

// Allocates the MultiParticle state once, on first use.
int MPEnsure(gomc_box *b) {
  MPState &mp = b->mp;
  if (mp.ready) return GOMC_OK;
  const size_t na = sizeof(double) * std::max(b->natoms, 1), nm = sizeof(double) * std::max(b->nmols, 1);
  bool ok = true;
  ok &= hipMalloc(&mp.xn, na) == hipSuccess;
  ok &= hipMalloc(&mp.yn, na) == hipSuccess;
  ok &= hipMalloc(&mp.zn, na) == hipSuccess;
  for (int s = 0; s < 2; ++s)
    for (int d = 0; d < 3; ++d) {
      ok &= hipMalloc(&mp.com[s][d], nm) == hipSuccess;
      ok &= hipMalloc(&mp.aF[s][d], na) == hipSuccess;
      ok &= hipMalloc(&mp.aFR[s][d], na) == hipSuccess;
      ok &= hipMalloc(&mp.mF[s][d], nm) == hipSuccess;
      ok &= hipMalloc(&mp.mFR[s][d], nm) == hipSuccess;
      ok &= hipMalloc(&mp.tq[s][d], nm) == hipSuccess;
    }
  for (int d = 0; d < 3; ++d) ok &= hipMalloc(&mp.tk[d], nm) == hipSuccess;
  ok &= hipMalloc(&mp.inRange, sizeof(int) * std::max(b->nmols, 1)) == hipSuccess;
  ok &= hipMalloc(&mp.wpart, sizeof(double) * ((b->nmols + kBlock - 1) / kBlock + 1)) == hipSuccess;
  ok &= hipMalloc(&mp.wcounter, sizeof(unsigned)) == hipSuccess;
  if (!ok) {
    MPFree(b);
    return Fail(b, GOMC_ERR_HIP, "MultiParticle allocation failed");
  }
  mp.molStart = b->molStartDev;  // owned by the box
  HIP_TRY(b, hipMemset(mp.wcounter, 0, sizeof(unsigned)));
  mp.ready = true;
  return GOMC_OK;
}

constexpr int kFailSlot = 15;  // of hostRes: a transform failed

// Arrays between the device and the box's staging memory, all of a call's in
// one launch: a copy command an array costs about 10 us each way for pageable
// memory, whatever its length (the 15 arrays and dozen waits of a force
// evaluation took 340 of 453 us for 1000 waters).
constexpr int kCopyMax = 6;
struct CopyArgs {
  const double *src[kCopyMax];
  double *dst[kCopyMax];
  int n[kCopyMax];
};
__global__ void __launch_bounds__(kBlock) CopyKernel(const CopyArgs a) {
  const int v = blockIdx.y, n = a.n[v];
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock)
    a.dst[v][i] = a.src[v][i];
}
static hipError_t LaunchCopies(const CopyArgs &a, int count, hipStream_t s) {
  int most = 1;
  for (int v = 0; v < count; ++v) most = std::max(most, a.n[v]);
  const int g = std::min((most + kBlock - 1) / kBlock, 256);
  hipLaunchKernelGGL(CopyKernel, dim3(g, count), dim3(kBlock), 0, s, a);
  return hipGetLastError();
}

// Device arrays to the host, one or two sets of three (a null destination is
// passed over); ends with the call's wait.
static int CopyOut(gomc_box *b, double *const *d0, double *const *s0, int n0,
                   double *const *d1 = nullptr, double *const *s1 = nullptr, int n1 = 0) {
  int rc = EnsureStage(b, 3 * (size_t(b->natoms) + 2 * size_t(b->nmols)));
  if (rc) return rc;
  CopyArgs a{};
  double *to[kCopyMax], *at = b->devStage;
  int count = 0;
  auto add = [&](double *const *d, double *const *s, int n) {
    for (int k = 0; k < 3; ++k)
      if (d[k]) {
        to[count] = d[k];
        a.src[count] = s[k];
        a.dst[count] = at;
        a.n[count++] = n;
        at += n;
      }
  };
  add(d0, s0, n0);
  if (d1) add(d1, s1, n1);
  if (count) HIP_TRY(b, LaunchCopies(a, count, b->stream));
  rc = Sync(b);
  if (rc) return rc;
  for (int v = 0; v < count; ++v)
    std::memcpy(to[v], b->stage + (a.dst[v] - b->devStage), sizeof(double) * a.n[v]);
  return GOMC_OK;
}

// The driver keeps the authoritative centres on the host; a MultiParticle
// step starts from them.  Not waited for: their place in the staging memory is
// behind what CopyOut returns, and every call that uploads them ends with a
// wait.
int MPUploadCom(gomc_box *b) {
  const size_t n = b->nmols, off = 3 * (size_t(b->natoms) + n);
  int rc = EnsureStage(b, off + 3 * n);
  if (rc) return rc;
  CopyArgs a{};
  const std::vector<double> *com[3] = {&b->comx, &b->comy, &b->comz};
  for (int d = 0; d < 3; ++d) {
    std::copy(com[d]->begin(), com[d]->begin() + n, b->stage + off + d * n);
    a.src[d] = b->devStage + off + d * n;
    a.dst[d] = b->mp.com[0][d];
    a.n[d] = b->nmols;
  }
  HIP_TRY(b, LaunchCopies(a, 3, b->stream));
  return GOMC_OK;
}

// Pair forces of the current coordinates into force set `set`; their energies
// are hostRes[0] and [1] after the caller's wait.
static int MPPairForce(gomc_box *b, int set) { return PairForces(b, b->mp.aF[set]); }

// Reciprocal forces of the current coordinates from the "new" sums; not waited
// for.
static int MPRecipForce(gomc_box *b, int set) {
  MPState &mp = b->mp;
  if (!b->ewald || !b->recipReady) {
    for (int d = 0; d < 3; ++d)
      HIP_TRY(b, hipMemsetAsync(mp.aFR[set][d], 0, sizeof(double) * b->natoms, b->stream));
    return GOMC_OK;
  }
  RecipForceArgs a;
  int rc = RecipForceParts(b, b->sumRnew, b->sumInew, &a.k);
  if (rc) return rc;
  a.g = b->geom;
  a.x = b->x;
  a.y = b->y;
  a.z = b->z;
  a.q = b->q;
  a.mol = b->mol;
  a.molStart = mp.molStart;
  a.natoms = b->natoms;
  a.fx = mp.aFR[set][0];
  a.fy = mp.aFR[set][1];
  a.fz = mp.aFR[set][2];
  hipLaunchKernelGGL(RecipForceKernel, dim3((b->natoms + kWave - 1) / kWave), dim3(kWave), 0,
                     b->stream, a);
  HIP_TRY(b, hipGetLastError());
  return GOMC_OK;
}

// Not waited for.
static int MolTerms(gomc_box *b, int set, int comSet, int mode) {
  MPState &mp = b->mp;
  MolTermsArgs a;
  a.g = b->geom;
  a.x = b->x;
  a.y = b->y;
  a.z = b->z;
  a.cx = mp.com[comSet][0];
  a.cy = mp.com[comSet][1];
  a.cz = mp.com[comSet][2];
  a.molStart = mp.molStart;
  a.nmols = b->nmols;
  a.mode = mode;
  for (int d = 0; d < 3; ++d) {
    a.aF[d] = mp.aF[set][d];
    a.aFR[d] = mp.aFR[set][d];
    a.mF[d] = mp.mF[set][d];
    a.mFR[d] = mp.mFR[set][d];
    a.tq[d] = mp.tq[set][d];
  }
  const int g = std::max(1, (b->nmols + kBlock - 1) / kBlock);
  hipLaunchKernelGGL(MolTermsKernel, dim3(g), dim3(kBlock), 0, b->stream, a);
  HIP_TRY(b, hipGetLastError());
  return GOMC_OK;
}

// Transform -> CalcEn -> GetCoeff (MultiParticle.h:332-511) on the
// reference force set; out = {inter, real, recip, w_ratio, fail}.  On
// success the trial coordinates are the box's current ones until
// MPAccept decides.
static int MPTrial(gomc_box *b, int rotate, uint64_t step, double max, double out[5]) {
  MPState &mp = b->mp;
  const int R = mp.ref, N = 1 - mp.ref;
  b->stageMol = -1;
  b->hostRes[kFailSlot] = 0.0;  // nothing of this box's runs: every call ends with a wait
  TransformArgs t;
  t.g = b->geom;
  t.nmols = b->nmols;
  t.rotate = rotate;
  t.step = step;
  t.seed = b->seed;
  t.beta = b->beta;
  t.max = max;
  t.x = b->x;
  t.y = b->y;
  t.z = b->z;
  t.cx = mp.com[0][0];
  t.cy = mp.com[0][1];
  t.cz = mp.com[0][2];
  t.xn = mp.xn;
  t.yn = mp.yn;
  t.zn = mp.zn;
  t.ncx = mp.com[1][0];
  t.ncy = mp.com[1][1];
  t.ncz = mp.com[1][2];
  t.molStart = mp.molStart;
  for (int d = 0; d < 3; ++d) {
    t.mF[d] = mp.mF[R][d];
    t.mFR[d] = mp.mFR[R][d];
    t.tq[d] = mp.tq[R][d];
    t.tk[d] = mp.tk[d];
  }
  t.inRange = mp.inRange;
  t.fail = b->devRes + kFailSlot;
  const int g = std::max(1, (b->nmols + kBlock - 1) / kBlock);
  hipLaunchKernelGGL(TransformKernel, dim3(g), dim3(kBlock), 0, b->stream, t);
  HIP_TRY(b, hipGetLastError());
  int rc = Sync(b);
  if (rc) return rc;
  const bool fail = b->hostRes[kFailSlot] != 0.0;
  out[0] = b->pot.inter;
  out[1] = b->pot.real;
  out[2] = b->pot.recip;
  out[3] = 1.0;
  out[4] = fail ? 1.0 : 0.0;
  if (fail) return GOMC_OK;
  // CalcEn on the trial coordinates: they become the box's coordinates.
  std::swap(b->x, mp.xn);
  std::swap(b->y, mp.yn);
  std::swap(b->z, mp.zn);
  for (int d = 0; d < 3; ++d) std::swap(mp.com[0][d], mp.com[1][d]);
  if (b->ewald) {
    rc = RecipSums(b, &out[2]);
    if (rc) return rc;
  }
  rc = MPPairForce(b, N);
  if (!rc) rc = MPRecipForce(b, N);
  if (!rc) rc = MolTerms(b, N, 0, 7);
  if (rc) return rc;
  CoeffArgs c;
  c.nmols = b->nmols;
  c.rotate = rotate;
  c.lBeta = kLambda * b->beta;
  c.max = max;
  for (int d = 0; d < 3; ++d) {
    c.tk[d] = mp.tk[d];
    c.nF[d] = mp.mF[N][d];
    c.nFR[d] = mp.mFR[N][d];
    c.nT[d] = mp.tq[N][d];
    c.oF[d] = mp.mF[R][d];
    c.oFR[d] = mp.mFR[R][d];
    c.oT[d] = mp.tq[R][d];
  }
  c.inRange = mp.inRange;
  c.parts = mp.wpart;
  c.counter = mp.wcounter;
  c.result = b->devRes + 4;
  hipLaunchKernelGGL(CoeffKernel, dim3(g), dim3(kBlock), 0, b->stream, c);
  HIP_TRY(b, hipGetLastError());
  rc = Sync(b);
  if (rc) return rc;
  out[0] = b->hostRes[0];
  out[1] = b->hostRes[1];
  double w = b->hostRes[4];
  out[3] = std::isfinite(w) ? w : 0.0;
  return GOMC_OK;
}

// MultiParticle::Accept's state change (MultiParticle.h:522-538).
static int MPAccept(gomc_box *b, bool result, bool evaluated, const double e[3]) {
  MPState &mp = b->mp;
  if (result) {
    b->pot.inter = e[0];
    b->pot.real = e[1];
    b->pot.recip = e[2];
    b->pot.Total();
    mp.ref = 1 - mp.ref;
    TrialCellsInvalidate(b);  // every molecule moved
    if (b->ewald) gomc_recip_accept(b);
    double *dx[3] = {b->hx.data(), b->hy.data(), b->hz.data()},
           *dc[3] = {b->comx.data(), b->comy.data(), b->comz.data()},
           *sx[3] = {b->x, b->y, b->z};
    int rc = CopyOut(b, dx, sx, b->natoms, dc, mp.com[0], b->nmols);
    // every molecule moved: EwaldCached::BoxReciprocalSums refilled the cache
    if (!rc && b->cached) rc = CacheBuild(b);
    return rc;
  }
  if (evaluated) {
    std::swap(b->x, mp.xn);
    std::swap(b->y, mp.yn);
    std::swap(b->z, mp.zn);
    for (int d = 0; d < 3; ++d) std::swap(mp.com[0][d], mp.com[1][d]);
  }
  return GOMC_OK;
}

// Prep's force evaluation (MultiParticle.h:207-230) for the current state.
static int MPPrepForces(gomc_box *b) {
  const int R = b->mp.ref;
  int rc = GOMC_OK;
  if (b->ewald) rc = gomc_recip_copy_ref_to_new(b);
  if (!rc) rc = MPRecipForce(b, R);
  if (!rc) rc = MPPairForce(b, R);
  if (!rc) rc = MolTerms(b, R, 0, 7);
  if (!rc) b->pot.Total();
  return rc;
}

// One MultiParticle move of the driver: Prep (the move type from MT19937,
// MultiParticle.h:176-182) -> Transform -> CalcEn -> Accept, with the
// acceptance draw from Philox counter N_mol (MultiParticle.h:521).
int MPMove(gomc_box *b, uint64_t step, int &moveType, int &accepted, int &failed, double dE[3]) {
  int rc = MPEnsure(b);
  if (!rc) rc = FlushPending(b);
  if (!rc) rc = MPUploadCom(b);
  if (rc) return rc;
  MPState &mp = b->mp;
  bool allTranslate = true;
  for (const auto &k : b->kindType) allTranslate = allTranslate && k.size() == 1;
  moveType = allTranslate ? 0 : int(b->mt.Below(1));
  if (mp.singleAccepted) {
    rc = MPPrepForces(b);
    if (rc) return rc;
  }
  const double max = moveType ? mp.rMax : mp.tMax;
  double out[5];
  rc = MPTrial(b, moveType, step, max, out);
  if (rc) return rc;
  const bool fail = out[4] != 0.0;
  Energies pn = b->pot;
  if (!fail) {
    pn.inter = out[0];
    pn.real = out[1];
    pn.recip = out[2];
  }
  const double uBoltz = std::exp(-b->beta * (pn.Total() - b->pot.Total()));
  const double accept = (fail ? 1.0 : out[3]) * uBoltz;
  const U64x4 r = Philox(uint64_t(uint32_t(b->nmols)), 0, 0, 0, step, b->seed);
  const double pr = U01(r.v[0]);
  const bool result = !fail && pr < accept;
  for (int i = 0; i < 3; ++i) dE[i] = fail ? 0.0 : out[i] - (i == 0 ? b->pot.inter : i == 1 ? b->pot.real : b->pot.recip);
  rc = MPAccept(b, result, !fail, out);
  if (rc) return rc;
  mp.itries[moveType]++;
  if (result) mp.iacc[moveType]++;
  mp.singleAccepted = false;
  accepted = result;
  failed = fail;
  return GOMC_OK;
}

}  // namespace gomc

// ====================================================================== C ABI
extern "C" {

int gomc_box_force(gomc_box *b, double *lj, double *real, double *afx, double *afy, double *afz,
                   double *mfx, double *mfy, double *mfz) {
  if (!b || !lj || !real) return GOMC_ERR_ARG;
  (void)hipSetDevice(b->device);
  int rc = MPEnsure(b);
  if (!rc) rc = FlushPending(b);
  if (!rc) rc = MPPairForce(b, b->mp.ref);
  if (!rc) rc = MolTerms(b, b->mp.ref, 0, 1);
  if (rc) return rc;
  double *da[3] = {afx, afy, afz}, *dm[3] = {mfx, mfy, mfz};
  rc = CopyOut(b, da, b->mp.aF[b->mp.ref], b->natoms, dm, b->mp.mF[b->mp.ref], b->nmols);
  if (rc) return rc;
  *lj = b->hostRes[0];
  *real = b->hostRes[1];
  return GOMC_OK;
}

int gomc_box_force_recip(gomc_box *b, double *afx, double *afy, double *afz, double *mfx,
                         double *mfy, double *mfz) {
  if (!b) return GOMC_ERR_ARG;
  (void)hipSetDevice(b->device);
  int rc = MPEnsure(b);
  if (!rc) rc = FlushPending(b);
  if (!rc) rc = MPRecipForce(b, b->mp.ref);
  if (!rc) rc = MolTerms(b, b->mp.ref, 0, 2);
  if (rc) return rc;
  double *da[3] = {afx, afy, afz}, *dm[3] = {mfx, mfy, mfz};
  return CopyOut(b, da, b->mp.aFR[b->mp.ref], b->natoms, dm, b->mp.mFR[b->mp.ref], b->nmols);
}

int gomc_torque(gomc_box *b, double *tx, double *ty, double *tz) {
  if (!b) return GOMC_ERR_ARG;
  (void)hipSetDevice(b->device);
  int rc = MPEnsure(b);
  if (!rc) rc = FlushPending(b);
  if (!rc) rc = MPUploadCom(b);
  if (!rc) rc = MolTerms(b, b->mp.ref, 0, 4);
  if (rc) return rc;
  double *dt[3] = {tx, ty, tz};
  return CopyOut(b, dt, b->mp.tq[b->mp.ref], b->nmols);
}

int gomc_mp_trial(gomc_box *b, int move_type, uint64_t step, double max, double out[5]) {
  if (!b || !out || (move_type != 0 && move_type != 1) || !(max > 0.0)) return GOMC_ERR_ARG;
  (void)hipSetDevice(b->device);
  int rc = MPEnsure(b);
  if (!rc) rc = FlushPending(b);
  if (!rc) rc = MPUploadCom(b);
  if (!rc) rc = MPTrial(b, move_type, step, max, out);
  return rc;
}

int gomc_mp_accept(gomc_box *b, int accept, const double out[5]) {
  if (!b || !out || !b->mp.ready) return GOMC_ERR_ARG;
  (void)hipSetDevice(b->device);
  const bool fail = out[4] != 0.0;
  if (accept && fail) return Fail(b, GOMC_ERR_STATE, "cannot accept a failed transform");
  int rc = MPAccept(b, accept != 0, !fail, out);
  if (!rc) b->mp.singleAccepted = false;
  return rc;
}

int gomc_mp_settings(const gomc_box *b, double out[2]) {
  if (!b || !out) return GOMC_ERR_ARG;
  out[0] = b->mp.tMax;
  out[1] = b->mp.rMax;
  return GOMC_OK;
}

}  // extern "C"
