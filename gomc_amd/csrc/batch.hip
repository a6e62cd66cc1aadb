// Batched persistent MC on gfx950: a 1024-thread workgroup runs the boxes
// of its task list one after another, making all of a box's moves of a
// launch without leaving the kernel; a large box is run by a team of 2, 4
// or 8 workgroups that split its pair items and k-vectors and exchange
// partial sums once per pass.  Per move: Philox draws (made 64 moves ahead,
// one lane each), the trial coordinates (Translate/Rotate,
// src/Coordinates.cpp:83-128), the pair-energy change over every other
// molecule (MoleculeInter, src/CalculateEnergy.cpp:581-686), the
// structure-factor change per k-vector (MolReciprocal,
// src/Ewald.cpp:409-473), the Metropolis test (src/moves/Translate.h:97-138)
// and, on acceptance, the update of coordinates and S(k).
//
// A pass holds two moves where it can (an even step A and the odd step B after
// it): B's sums are found for A kept and for A moved, and whichever holds is
// taken when A is decided.  One move alone is bound by its chain of waits
// (draws to tables, tables to phases, sums to decision) and its reciprocal
// half reads all of S(k) for one molecule; two share both.  The chain is the
// same whether the moves share a pass or not, to the bit (CrossTerms), so a
// run's results do not depend on where launches cut it.
//
// Phases e^{i k.r} come from per-dimension tables e^{i (c_d n) r_d},
// n = 0..nmax, built each pass for the moving molecules' old and new
// positions (one sincos per table entry), and advanced along nz.
//
// What bounds it: over a cycle of 256 boxes a SIMD issues a vector instruction in
// 38 % of its cycles and a wave waits two thirds of its own, at the passes'
// barriers and for memory; within the pair and reciprocal phases fewer
// instructions are fewer microseconds.  Measured on MI355X, rigid 3-site water,
// microseconds a move of one box alone, FP64 / mixed, against one move a pass,
// libm-free erfc by polynomial and FP64 centre tests:
//   202 waters, 1 workgroup     7.9 /  7.3, was 10.4 /  9.4
//   500                         8.9 /  8.2, was 13.3 / 12.3
//   985                         9.8 /  8.8, was 14.4 / 12.9
//   1700                       11.6 / 10.4, was 16.1 / 14.1
//   2454, team of 2             9.8 /  8.0, was 13.7 / 12.2
//   3950, team of 8             8.1 /  6.3, was 11.0 / 10.3
// A launch itself costs 10 us more in the kernel: a workgroup loads its box's
// pointers, Coulomb table and two programs.  The calls are shorter all the same
// (one box of 300 waters, 1 / 4 / 40 moves 76 / 104 / 479 us, was 80 / 115 / 540):
// the host copies and waits less.
#include "batch.hpp"
#include "coul_table.hpp"
#include "device_common.hpp"

namespace gomc {
namespace {

// Pointers into global memory (HBM) and LDS.  The phases are out-of-line
// functions; a plain pointer parameter there is a generic (flat) address,
// and every flat access also counts against the LDS wait counter, so a
// wait for an LDS read would stall on outstanding HBM loads.
#define GMEM __attribute__((address_space(1)))
#define LMEM __attribute__((address_space(3)))
template <typename T>
__device__ __forceinline__ GMEM T *Gp(T *p) {
  return (GMEM T *)p;
}
template <typename T>
__device__ __forceinline__ LMEM T *Lp(T *p) {
  return (LMEM T *)p;
}

// Phase-table entries: FP64 in the FP64 mode, FP32 in the mixed mode.
template <typename T>
struct CplxT {
  T re, im;
};
using Cplx = CplxT<double>;

template <typename T>
__device__ __forceinline__ CplxT<T> CMul(CplxT<T> a, CplxT<T> b) {
  return {fma(a.re, b.re, -(a.im * b.im)), fma(a.re, b.im, a.im * b.re)};
}

// Precision traits: P = 0 FP64 everywhere; P = 1 FP32 pair terms and phase
// products (distances, accumulation, S(k), totals and the Metropolis
// exponent stay FP64).
template <int P>
struct Prec {
  using T = double;
};
template <>
struct Prec<1> {
  using T = float;
};

// One proposed move of a pass.
struct MoveOne {
  double oldp[3][kBatchMaxAtoms], newp[3][kBatchMaxAtoms];
  double rel[2][kBatchMaxAtoms][4];  // old and new atoms from their centre (minimum image); pad
  double com[2][3];                  // old and new centre
  int mol, type;
};

// Sums of a pass over its two moves A and B (kNumSums words, exchanged as 16).
// kX...: molecule A against B where A stays (0) or has moved (1).
enum : int {
  kLjA, kRealA, kLjB, kRealB, kOvA, kOvB,  // by the pair waves
  kRecA, kRecB0, kRecB1,                   // by the reciprocal waves; B after A stayed / moved
  kXLj0, kXReal0, kXOv0, kXLj1, kXReal1, kXOv1,  // by one pair wave
  kNumSums
};
static_assert(kNumSums <= kXchgVals, "a pass's sums fit the exchange block");

struct alignas(16) MoveShared {
  MoveOne mv[2];
  double red[kBatchThreads / kWave][kXchgVals], tot[kXchgVals];
  int accept[2];
  int abort;  // a team exchange ran out of time: the box stops
};

// A value every lane holds alike, moved to scalar registers.
__device__ __forceinline__ double Uniform(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_readfirstlane(uint32_t(u));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(uint32_t(u >> 32));
  return __builtin_bit_cast(double, (uint64_t(hi) << 32) | lo);
}
__device__ __forceinline__ float Uniform(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(uint32_t, v)));
}

__device__ __forceinline__ int64_t UniformI64(int64_t v) {
  const uint64_t u = uint64_t(v);
  const uint32_t lo = __builtin_amdgcn_readfirstlane(uint32_t(u));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(uint32_t(u >> 32));
  return int64_t((uint64_t(hi) << 32) | lo);
}

template <typename T>
__device__ __forceinline__ GMEM T *UniformPtr(GMEM T *p) {
  return (GMEM T *)UniformI64((int64_t)p);
}

// d by its minimum image: d - L rint(d / L).
__device__ __forceinline__ double Image(double d, double L, double inv) {
  return fma(-L, rint(d * inv), d);
}

// One phase-table entry: e^{i (c_d n) r}.  FP64: in half-turns, n (2 r / L),
// whose reduction is exact and short.
template <typename T>
__device__ __forceinline__ CplxT<T> PhaseEntry(const LMEM BatchBox *sb, int d, int n, double r) {
  if constexpr (sizeof(T) == 8) {
    double sn, c;
    sincospi(double(n) * (r * sb->twoInvL[d]), &sn, &c);
    return {c, sn};
  } else {
    // FP64 reduction to [-pi, pi), FP32 sincos of the remainder.
    const double ang = (sb->kc[d] * double(n)) * r;
    const double turns = ang * (0.5 * M_1_PI);
    const float red = float((turns - rint(turns)) * (2.0 * M_PI));
    float sn, c;
    sincosf(red, &sn, &c);
    return {c, sn};
  }
}

// MoveSettings::AdjustMoves (src/MoveSettings.cpp:148-258), by one lane.
__device__ __noinline__ void Adjust(const LMEM BatchBox *sb, LMEM BatchState *st) {
  const double lmin = fmin(sb->L[0], fmin(sb->L[1], sb->L[2]));
  for (int t = 0; t < 2; ++t) {
    if (st->tempTries[t] > 0) {
      const double acc = double(st->tempAccepted[t]) / double(st->tempTries[t]);
      const double fract = acc / 0.5;
      st->scale[t] *= (fract > 0.0) ? fract : 0.5;
    }
    const double lo = t == 0 ? 1.0e-10 : 1.0e-6;
    const double hi = t == 0 ? (lmin * 0.5) - 1.0e-7 : M_PI - 1.0e-7;
    st->scale[t] = fmin(fmax(st->scale[t], lo), hi);
    st->tempTries[t] = 0;
    st->tempAccepted[t] = 0;
  }
}

// The molecule a draw picks.
__device__ __forceinline__ int PickMol(double u1, int nmols) {
  const int m = int(u1 * nmols);
  return m >= nmols ? nmols - 1 : m;
}

// Lane p of a move's lanes: the move's kind, molecule and shift or rotation
// (every lane makes the same ones), then the old and new position of atom p
// (Translate/Rotate, src/Coordinates.cpp:83-128).
__device__ __noinline__ void Propose(const LMEM BatchBox *sb, const LMEM BatchState *st,
                                     LMEM MoveOne *mv, const LMEM double *u, int p,
                                     const GMEM double *X, const GMEM double *Y,
                                     const GMEM double *Z, const GMEM double *CX,
                                     const GMEM double *CY, const GMEM double *CZ) {
  const int len = sb->molLen, m = PickMol(u[1], sb->nmols);
  const int t = (len <= 1 || u[0] < sb->pDisp) ? 0 : 1;
  const int64_t ai = int64_t(m) * len + p;
  const double o[3] = {X[ai], Y[ai], Z[ai]}, com[3] = {CX[m], CY[m], CZ[m]};
  double nw[3], ncom[3] = {com[0], com[1], com[2]};  // a rotation keeps the centre
  if (t == 0) {
    const double bb = st->scale[0], b2 = 2.0 * bb;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double sh = u[2 + d] * b2 - bb;
      ncom[d] = Wrap(com[d] + sh, sb->L[d]);
      nw[d] = Wrap(o[d] + sh, sb->L[d]);
    }
  } else {
    const double bb = st->scale[1];
    const double theta = u[2] * (2.0 * bb) - bb;
    const double cu = u[3] * 2.0 - 1.0;
    const double root = sqrt(1.0 - cu * cu);
    const double sp = u[6], cp = u[7];  // sincos(2 pi u[4]), made with the draws
    const double ax[3] = {root * cp, root * sp, cu};
    double sn, c;
    sincos(theta, &sn, &c);
    const double cr[3][3] = {{0.0, -ax[2], ax[1]}, {ax[2], 0.0, -ax[0]}, {-ax[1], ax[0], 0.0}};
    double v[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) v[d] = Unwrap(o[d], com[d], sb->L[d], sb->half[d]) + (-com[d]);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      double rot[3];
#pragma unroll
      for (int j = 0; j < 3; ++j)
        rot[j] = (i == j ? c : 0.0) + (sn * cr[i][j] + (1 - c) * (ax[i] * ax[j]));
      const double r = rot[0] * v[0] + rot[1] * v[1] + rot[2] * v[2];
      nw[i] = Wrap(r + com[i], sb->L[i]);
    }
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    mv->oldp[d][p] = o[d];
    mv->newp[d][p] = nw[d];
    mv->rel[0][p][d] = MinImage(o[d] - com[d], sb->L[d], sb->half[d]);
    mv->rel[1][p][d] = MinImage(nw[d] - ncom[d], sb->L[d], sb->half[d]);
  }
  if (p == 0) {
    mv->mol = m;
    mv->type = t;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      mv->com[0][d] = com[d];
      mv->com[1][d] = ncom[d];
    }
  }
}

// Philox draws of one move: u[0..5] (two blocks, counter {step, 0|1}), and
// sin, cos of a rotation's axis azimuth 2 pi u[4] in u[6], u[7] (a function
// of the draw alone, so made here, 64 moves ahead, not by thread 0 within
// the move).
__device__ __noinline__ void MoveDraws(uint64_t seed, uint64_t step, LMEM double *out) {
  const U64x4 r0 = Philox(step, 0, 0, 0, seed, kPhiloxTag);
  const U64x4 r1 = Philox(step, 1, 0, 0, seed, kPhiloxTag);
  out[0] = U01(r0.v[0]);
  out[1] = U01(r0.v[1]);
  out[2] = U01(r0.v[2]);
  out[3] = U01(r0.v[3]);
  out[4] = U01(r1.v[0]);
  out[5] = U01(r1.v[1]);
  const double phi = out[4] * (2.0 * M_PI);
  double sn, c;
  sincos(phi, &sn, &c);
  out[6] = sn;
  out[7] = c;
}

// Phase tables e^{i (c_d n) r_d}, n = 0..nmax_d, for the moving molecules' old
// (pos < len) and new positions; one entry per thread-iteration.
template <typename T>
using PhaseTab = CplxT<T>[2 * kBatchMaxAtoms][3][kBatchMaxN + 1];

template <typename T>
__device__ __forceinline__ void BuildTables(const LMEM BatchBox *sb, const LMEM MoveOne *mv, int len,
                                         int first, int moves, LMEM PhaseTab<T> *tab) {
  const int n0 = sb->nmax[0] + 1, n1 = sb->nmax[1] + 1, per = n0 + n1 + sb->nmax[2] + 1;
  for (int e = threadIdx.x; e < moves * 2 * len * per; e += kBatchThreads) {
    const int mp = e / per, m = first + mp / (2 * len), pos = mp % (2 * len);
    int rem = e - mp * per, d = 0;
    if (rem >= n0) {
      rem -= n0;
      d = 1;
      if (rem >= n1) {
        rem -= n1;
        d = 2;
      }
    }
    const double r = pos < len ? mv[m].oldp[d][pos] : mv[m].newp[d][pos - len];
    const CplxT<T> c = PhaseEntry<T>(sb, d, rem, r);
    tab[m][pos][d][rem].re = c.re;
    tab[m][pos][d][rem].im = c.im;
  }
}

// Per-wave queues of in-cutoff pairs, one for each move of a pass: squared
// distance and a code (pair-table index | new-position flag << 8).
struct PairQueue {
  double d2[2][2 * kWave];
  uint16_t code[2][2 * kWave];
};

struct LjReal {
  double lj, real;
};

// The box's Coulomb table (coul_table.hpp), copied to LDS when its run starts.
struct alignas(16) CoulTab {
  double c[kTabWords];
};

// The same factor below the table's first octave.
__device__ __noinline__ double CoulFactor(const LMEM BatchBox *sb, double d2) {
  const double r = sqrt(d2);
  return sb->ewald ? erfc(sb->alpha * r) / r : 1.0 / r;
}

// Energy terms of one pair (FFParticle::CalcEn / CalcCoulomb,
// src/FFParticle.cpp:295-399), signed: + new position, - old position.
// n = 12 (checked at setup): repulsion = attraction^2.
template <typename T>
__device__ __forceinline__ LjReal PairTerm(const LMEM BatchBox *sb, const LMEM CoulTab *tab,
                                           double d2, int code) {
  LjReal out{0.0, 0.0};
  const int pq = code & 0xff;
  const double sign = (code >> 8) ? 1.0 : -1.0;
  const double qiqj = sb->qq[pq], eps = sb->epsCn[pq];
  if constexpr (sizeof(T) == 8) {
    if (sb->elect && qiqj != 0.0 && !(sb->rCutCoulSq < d2)) {
      double t;
      const int row = TabRow(d2, sb->tabBase, &t);
      const double f = uint32_t(row) < uint32_t(kTabRows)
                           ? TabValue((const LMEM TabPair *)tab->c, (const LMEM double *)tab->c, row, t)
                           : CoulFactor(sb, d2);
      out.real = (sign * qiqj) * f;
    }
    if (eps != 0.0 && !(sb->rCutLJSq < d2)) {
      double ir2 = __builtin_amdgcn_rcp(d2);  // two Newton steps
      ir2 = fma(ir2, fma(-d2, ir2, 1.0), ir2);
      ir2 = fma(ir2, fma(-d2, ir2, 1.0), ir2);
      const double rRat2 = sb->sigSq[pq] * ir2;
      const double att = rRat2 * rRat2 * rRat2;
      out.lj = sign * (eps * (att * att - att));
    }
  } else {
    if (sb->elect && qiqj != 0.0 && !(sb->rCutCoulSq < d2)) {
      const T dist = sqrt(T(d2));
      const T ec = sb->ewald ? T(qiqj) * erfc(T(sb->alpha) * dist) / dist : T(qiqj) / dist;
      out.real = sign * double(ec);
    }
    if (eps != 0.0 && !(sb->rCutLJSq < d2)) {
      const T rRat2 = T(sb->sigSq[pq]) / T(d2);
      const T att = rRat2 * rRat2 * rRat2;
      out.lj = sign * double(T(eps) * (att * att - att));
    }
  }
  return out;
}

// The terms of this lane's queued pair, zero where `on` is false.
template <typename T>
__device__ __noinline__ LjReal QueuedPair(const LMEM BatchBox *sb, const LMEM CoulTab *tab,
                                          double d2, int code, bool on) {
  return on ? PairTerm<T>(sb, tab, d2, code) : LjReal{0.0, 0.0};
}

// The pair phase and the reciprocal phase of a pass are independent once the
// trial coordinates and phase tables exist, and neither fills the SIMDs alone
// (the pair phase waits on gathers and queues, the reciprocal phase on S(k)): waves 0 .. sb.pairWaves-1 run the pair phase while the
// other sb.kWidth threads run the reciprocal phase, with no barrier inside
// either.  A pass holds one move or two: B's energies are found for both
// outcomes of A, so the two share every latency and the S(k) traffic.

// Pair-energy changes of a pass (MoleculeInter, src/CalculateEnergy.cpp:
// 581-686), by the waves of the pair group.  Each wave takes its share of the
// (team member's) molecules, 64 at a time.  Level 1 (boxes with sb.cull): a
// molecule whose centre is at least rc + 2 r_max from both the old and the
// new centre of a moving molecule (minimum image) holds no pair inside the
// cutoff with it (triangle inequality); the centres are tested in FP32 with a
// margin that covers their rounding, and near molecules are listed per move.
// Level 2: whenever a list holds a wave's worth of atoms, one atom of a near
// molecule (of every other molecule without the cull) per lane is tested
// against the old and new positions of the moving atoms; distances inside the
// cutoff are compacted into the move's queue (ballot + prefix count) and
// their energies evaluated 64 at a time, so the erfc path runs with full
// waves.
//
// `skip`: the molecule the previous (even) step moved, left out of the odd
// step's sum and added by CrossTerms, whether the two steps share a pass or
// not; so a move's sum has the same terms in the same order in both.
template <typename T, int LEN, typename ComPtr>
__device__ __forceinline__ void PairPhase(const LMEM BatchBox *sb, const LMEM CoulTab *ctab,
                                       const LMEM MoveOne *mv,
                                       const GMEM double *X, const GMEM double *Y,
                                       const GMEM double *Z, ComPtr CX, ComPtr CY, ComPtr CZ,
                                       int nmols, int rank, int team, int has, int skip,
                                       LMEM PairQueue *queues, LMEM int *nearList,
                                       LMEM double *red) {
  constexpr int len = LEN, kPer = kWave / LEN;  // molecules a wave takes at once
  struct {
    double L[3];
  } g;
  double inv[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    g.L[d] = Uniform(sb->L[d]);
    inv[d] = Uniform(0.5 * sb->twoInvL[d]);
  }
  const bool wide = __builtin_amdgcn_readfirstlane(sb->wide) != 0;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);  // < pairWaves
  const int pw = __builtin_amdgcn_readfirstlane(sb->pairWaves);
  LMEM PairQueue *q = queues + wave;
  LMEM int *list[2] = {nearList + wave * 2 * kNearListLen, nearList + (wave * 2 + 1) * kNearListLen};
  const uint64_t below = (uint64_t(1) << lane) - 1;
  const bool cull = __builtin_amdgcn_readfirstlane(sb->cull) != 0;
  // an overlap is a pair inside the cutoff as well, however large RcutLow
  const double rCutSq = Uniform(sb->rCutSq), rLowSq = fmin(Uniform(sb->rCutLowSq), rCutSq);
  const uint32_t liveBits = __builtin_amdgcn_readfirstlane(uint32_t(sb->live));
  const int mol[2] = {__builtin_amdgcn_readfirstlane(mv[0].mol),
                      __builtin_amdgcn_readfirstlane(mv[1].mol)};
  float fL[3], fI[3], fo[2][3], fn[2][3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    fL[d] = Uniform(float(g.L[d]));
    fI[d] = Uniform(1.0f / fL[d]);
#pragma unroll
    for (int v = 0; v < 2; ++v) {
      fo[v][d] = Uniform(float(mv[v].com[0][d]));
      fn[v][d] = Uniform(float(mv[v].com[1][d]));
    }
  }
  const float nearSq = sb->nearCutSqF;
  int nnear[2] = {0, 0}, qn[2] = {0, 0};  // wave-uniform
  double lj[2] = {0.0, 0.0}, real[2] = {0.0, 0.0};
  uint64_t low[2] = {0, 0};  // lanes that saw an atom inside RcutLow of a new position
  auto far2 = [&](const float a[3], float x, float y, float z) {
    float dx = a[0] - x, dy = a[1] - y, dz = a[2] - z;
    dx = fmaf(-fL[0], rintf(dx * fI[0]), dx);
    dy = fmaf(-fL[1], rintf(dy * fI[1]), dy);
    dz = fmaf(-fL[2], rintf(dz * fI[2]), dz);
    return fmaf(dz, dz, fmaf(dy, dy, dx * dx));
  };
  const int k = lane / len, qa = lane - k * len;
  // level 2 for the last n listed molecules of move v (n <= kPer).  Where half
  // the box holds the cutoff and a molecule's radius (sb.wide), an atom's image
  // nearest the moving centre is also nearest every moving atom if it is
  // inside the cutoff of one: the image is found once per centre.
  // The loop over moving atoms is kept a loop and the evaluation inline: one
  // copy of it, and no call to save registers around.
  auto tests = [&](int v, int n, double xj, double yj, double zj) {
    const bool valid = lane < n * len;
    LMEM double *qd = q->d2[v];
    LMEM uint16_t *qc = q->code[v];
    int count = qn[v];
    double sl = 0.0, sr = 0.0;
#pragma unroll 1
    for (int isNew = 0; isNew < 2; ++isNew) {
      const LMEM double *com = mv[v].com[isNew];
      const double rx = Image(xj - com[0], g.L[0], inv[0]), ry = Image(yj - com[1], g.L[1], inv[1]),
                   rz = Image(zj - com[2], g.L[2], inv[2]);
#pragma unroll 1
      for (int p = 0; p < len; ++p) {
        const LMEM double *rel = mv[v].rel[isNew][p];
        double dx = rel[0] - rx, dy = rel[1] - ry, dz = rel[2] - rz;
        if (!wide) {
          dx = Image(dx, g.L[0], inv[0]);
          dy = Image(dy, g.L[1], inv[1]);
          dz = Image(dz, g.L[2], inv[2]);
        }
        const double d2 = fma(dz, dz, fma(dy, dy, dx * dx));
        if (isNew) low[v] |= __ballot(valid && d2 < rLowSq);
        const int pq = p * kBatchMaxAtoms + qa;
        const bool push = valid && ((liveBits >> pq) & 1) && rCutSq > d2;
        const uint64_t mask = __ballot(push);
        const int slot = __builtin_amdgcn_mbcnt_hi(
            uint32_t(mask >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(mask), uint32_t(count)));
        if (push) {
          qd[slot] = d2;
          qc[slot] = uint16_t(pq | (isNew << 8));
        }
        count += __popcll(mask);
        if (count >= kWave) {  // evaluate one full wave of pairs
          __builtin_amdgcn_wave_barrier();
          const LjReal t = PairTerm<T>(sb, ctab, qd[lane], qc[lane]);
          sl += t.lj;
          sr += t.real;
          const double d2n = qd[kWave + lane];
          const uint16_t cn = qc[kWave + lane];
          __builtin_amdgcn_wave_barrier();
          qd[lane] = d2n;
          qc[lane] = cn;
          count -= kWave;
          __builtin_amdgcn_wave_barrier();
        }
      }
    }
    qn[v] = count;
    lj[v] += sl;
    real[v] += sr;
  };
  const int mper = (nmols + team - 1) / team;
  const int t0 = rank * mper, t1 = min(nmols, t0 + mper);
  const int share = (max(t1 - t0, 0) + pw - 1) / pw;
  const int m0 = t0 + wave * share, m1 = min(t1, m0 + share);
  for (int base = m0;; base += kWave) {
    const bool last = base + kWave >= m1;
    const int j = base + lane;
    bool near[2] = {false, false};
    if (j < m1) {
      if (cull) {
        const float cx = CX[j], cy = CY[j], cz = CZ[j];
#pragma unroll
        for (int v = 0; v < 2; ++v)
          near[v] = far2(fo[v], cx, cy, cz) < nearSq || far2(fn[v], cx, cy, cz) < nearSq;
      } else {
        near[0] = near[1] = true;
      }
      near[0] = near[0] && (has & 1) && j != mol[0];
      near[1] = near[1] && (has & 2) && j != mol[1] && j != skip;
    }
#pragma unroll
    for (int v = 0; v < 2; ++v) {
      const uint64_t nmask = __ballot(near[v]);
      if (near[v]) list[v][nnear[v] + __popcll(nmask & below)] = j;
      nnear[v] += __popcll(nmask);
    }
    __builtin_amdgcn_wave_barrier();
    // both moves' atoms are loaded before either is tested
    while (nnear[0] >= kPer || nnear[1] >= kPer || (last && nnear[0] + nnear[1] > 0)) {
      double x[2] = {0.0, 0.0}, y[2] = {0.0, 0.0}, z[2] = {0.0, 0.0};
      int n[2];
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        n[v] = (last || nnear[v] >= kPer) ? min(nnear[v], kPer) : 0;
        nnear[v] -= n[v];
        if (lane < n[v] * len) {
          const uint32_t jj = 8u * uint32_t(list[v][nnear[v] + k] * len + qa);  // bytes
          x[v] = *(const GMEM double *)((const GMEM char *)X + jj);
          y[v] = *(const GMEM double *)((const GMEM char *)Y + jj);
          z[v] = *(const GMEM double *)((const GMEM char *)Z + jj);
        }
      }
      __builtin_amdgcn_wave_barrier();
      if (n[0] > 0) tests(0, n[0], x[0], y[0], z[0]);
      if (n[1] > 0) tests(1, n[1], x[1], y[1], z[1]);
    }
    if (last) break;
  }
  __builtin_amdgcn_wave_barrier();
  // the rest of both queues: A's pairs from lane 0 up, B's from lane 63 down
  // (the same lanes whether or not the other is there), together if they fit
  {
    const int b = kWave - 1 - lane;  // B's entry of this lane
    const bool together = qn[0] + qn[1] <= kWave;
    const bool isA = lane < qn[0];
    if (qn[0] > 0 || (together && qn[1] > 0)) {
      const bool isB = together && b < qn[1];
      const double d2 = isA ? q->d2[0][lane] : q->d2[1][isB ? b : 0];
      const int code = isA ? q->code[0][lane] : q->code[1][isB ? b : 0];
      const LjReal t = QueuedPair<T>(sb, ctab, d2, code, isA || isB);
      lj[0] += isA ? t.lj : 0.0;
      real[0] += isA ? t.real : 0.0;
      lj[1] += isA ? 0.0 : t.lj;
      real[1] += isA ? 0.0 : t.real;
    }
    if (!together) {
      const LjReal t = QueuedPair<T>(sb, ctab, q->d2[1][b], q->code[1][b], b < qn[1]);
      lj[1] += t.lj;
      real[1] += t.real;
    }
  }
  const double s0 = WaveSumDpp(lj[0]), s1 = WaveSumDpp(real[0]), s2 = WaveSumDpp(lj[1]),
               s3 = WaveSumDpp(real[1]);
  const bool oA = low[0] != 0, oB = low[1] != 0;
  if (lane == kWave - 1) {
    LMEM double *r = red + wave * kXchgVals;
    r[kLjA] = s0;
    r[kRealA] = s1;
    r[kLjB] = s2;
    r[kRealB] = s3;
    r[kOvA] = oA ? 1.0 : 0.0;
    r[kOvB] = oB ? 1.0 : 0.0;
  }
}

// The moving molecule B against molecule A (the one the even step before it
// moved), which its PairPhase sum leaves out: with A at its position before
// its move and, where A's move shares the pass, after it.  Run by one wave of
// one team member; a lane takes one (atom of B, atom of A, B old or new, A old
// or new).  Sums to red.
template <typename T>
__device__ __noinline__ void CrossTerms(const LMEM BatchBox *sb, const LMEM CoulTab *ctab,
                                        const LMEM MoveOne *mv,
                                        const GMEM double *X, const GMEM double *Y,
                                        const GMEM double *Z, int len, int has, int skip,
                                        LMEM double *red) {
  const int lane = threadIdx.x & (kWave - 1);
  const int sq = len * len, f = lane / sq, r = lane - f * sq, p = r / len, qa = r - p * len;
  const bool newB = f & 1, newA = f & 2;
  LjReal t{0.0, 0.0};
  bool ov = false;
  if (skip >= 0 && f < (has == 3 ? 4 : 2)) {
    double a[3], d[3];
    const int64_t ai = int64_t(skip) * len + qa;
    if (has == 3) {
#pragma unroll
      for (int i = 0; i < 3; ++i) a[i] = newA ? mv[0].newp[i][qa] : mv[0].oldp[i][qa];
    } else {
      a[0] = X[ai];
      a[1] = Y[ai];
      a[2] = Z[ai];
    }
#pragma unroll
    for (int i = 0; i < 3; ++i)
      d[i] = Image((newB ? mv[1].newp[i][p] : mv[1].oldp[i][p]) - a[i], sb->L[i],
                   0.5 * sb->twoInvL[i]);
    const double d2 = fma(d[2], d[2], fma(d[1], d[1], d[0] * d[0]));
    const int pq = p * kBatchMaxAtoms + qa;
    const bool inCut = sb->rCutSq > d2;
    ov = newB && inCut && d2 < sb->rCutLowSq;
    t = QueuedPair<T>(sb, ctab, d2, pq | (newB ? 256 : 0), inCut && ((sb->live >> pq) & 1));
  }
  // A's later position on the lanes of its earlier one, so that a sum has the
  // same order whichever of them holds the molecule's place
  const double ljN = __shfl(t.lj, lane + 2 * sq), realN = __shfl(t.real, lane + 2 * sq);
  const bool first = lane < 2 * sq, both = first && has == 3;
  const double l0 = WaveSumDpp(first ? t.lj : 0.0), r0 = WaveSumDpp(first ? t.real : 0.0),
               l1 = WaveSumDpp(both ? ljN : 0.0), r1 = WaveSumDpp(both ? realN : 0.0);
  const bool o0 = __any(ov && !newA), o1 = __any(ov && newA);
  if (lane == kWave - 1) {
    red[kXLj0] = l0;
    red[kXReal0] = r0;
    red[kXOv0] = o0 ? 1.0 : 0.0;
    red[kXLj1] = l1;
    red[kXReal1] = r1;
    red[kXOv1] = o1 ? 1.0 : 0.0;
  }
}

// Reciprocal-space energy changes of a pass (MolReciprocal,
// src/Ewald.cpp:409-473): per k-vector the change (dR, dI) of the structure
// factor and prefact * ((R+dR)^2 + (I+dI)^2 - R^2 - I^2), written as
// prefact * (dR (2R + dR) + dI (2I + dI)) so no large terms cancel; for the
// second move of a pass both from S and from S plus the first move's change.
// The changes are kept for the commit.
//
// A thread takes one segment of S k-vectors per round: consecutive nz at
// fixed (nx, ny).  The phase of each of the 2 LEN positions of a move is
// formed from the tables at the segment start, (ex * ey) * ez, and advanced
// along nz by one complex product with e^{i c_z z} per step, so a k-vector
// costs no table reads after the first of its segment.  The next k-vector's
// loads are issued before this one is worked on.
// pend, bit v: the last pass's move v was accepted and its change, still in
// the thread's slots, is added to S(k) here (Ewald::UpdateRecip,
// src/Ewald.cpp:1420) before the slots are reused.  Unused slots (kn -1, pref
// 0, S(k) 0) add zero.
constexpr int kZeroCode = (128 << 8) | (128 << 16);  // n = (0, 0, 0)

template <typename T>
__device__ __forceinline__ CplxT<T> TablePhase(const LMEM CplxT<T> (*row)[kBatchMaxN + 1], int code) {
  const int nx = code & 0xff;
  const int ny = ((code >> 8) & 0xff) - 128;
  const int nz = ((code >> 16) & 0xff) - 128;
  const LMEM CplxT<T> *px = &row[0][nx], *py = &row[1][ny < 0 ? -ny : ny],
                      *pz = &row[2][nz < 0 ? -nz : nz];
  CplxT<T> ex{px->re, px->im}, ey{py->re, py->im}, ez{pz->re, pz->im};
  if (ny < 0) ey.im = -ey.im;
  if (nz < 0) ez.im = -ez.im;
  return CMul(CMul(ex, ey), ez);
}

// The structure-factor changes of a pass's two moves; the second array is
// absent (null) where passes hold one move only.
struct DeltaPtrs {
  GMEM double *R[2], *I[2];
};

// Accumulates a + q b: one rounding in FP64, the product rounded on its own in
// FP32.
__device__ __forceinline__ double Axpy(double q, double b, double a) { return fma(q, b, a); }
__device__ __forceinline__ float Axpy(float q, float b, float a) { return a + q * b; }

// NM: moves of the pass; m0 the first (0: A or both, 1: B alone).  B of a pass
// of two uses the second delta arrays, a move alone the first.
//
// Loads and stores count down one counter in order, so a wait for a load also
// waits for the stores before it: every access of a step is unconditional
// (an unused slot's change and S(k) are zero and stay so) and two steps
// alternate between two sets of registers, which leaves a step's loads a whole
// step, and its stores two, before anything waits for them.
template <typename T, int S, int LEN, int NM>
__device__ __noinline__ void RecipPhase(const LMEM BatchBox *sb, const LMEM PhaseTab<T> *tab, int m0,
                                        const GMEM int32_t *kn0, const GMEM double *pref0,
                                        GMEM double *sumR0, GMEM double *sumI0, DeltaPtrs d0,
                                        int rank, int team, int pend, LMEM double *red) {
  const GMEM int32_t *kn = UniformPtr(kn0);
  const GMEM double *pref = UniformPtr(pref0);
  GMEM double *sumR = UniformPtr(sumR0), *sumI = UniformPtr(sumI0);
  GMEM double *dRa = UniformPtr(d0.R[0]), *dIa = UniformPtr(d0.I[0]);
  GMEM double *dRb = UniformPtr(d0.R[1]), *dIb = UniformPtr(d0.I[1]);
  rank = __builtin_amdgcn_readfirstlane(rank);
  team = __builtin_amdgcn_readfirstlane(team);
  pend = __builtin_amdgcn_readfirstlane(pend);
  m0 = __builtin_amdgcn_readfirstlane(m0);
  T q[LEN];
  CplxT<T> step[NM][2 * LEN];
#pragma unroll
  for (int p = 0; p < LEN; ++p)  // the same for every lane: kept in scalar registers
    q[p] = Uniform(fabs(sb->charge[p]) < 0.000000001 ? T(0) : T(sb->charge[p]));
#pragma unroll
  for (int v = 0; v < NM; ++v)
#pragma unroll
    for (int p = 0; p < 2 * LEN; ++p) {
      const LMEM CplxT<T> *c = &tab[m0 + v][p][2][1];
      step[v][p] = {Uniform(c->re), Uniform(c->im)};
    }
  double e0 = 0.0, e1 = 0.0, e2 = 0.0;  // the first move; the second after it stayed / moved
  // thread t of the reciprocal group owns column t of the W-wide layout
  const int W = __builtin_amdgcn_readfirstlane(sb->kWidth);
  const uint32_t t = threadIdx.x - uint32_t(__builtin_amdgcn_readfirstlane(sb->pairWaves)) * kWave;
  const int rounds = __builtin_amdgcn_readfirstlane(sb->kChunk);
  const int mine = rounds > rank ? (rounds - rank - 1) / team + 1 : 0;  // a member's rounds
  const int total = mine * S;
  CplxT<T> e[NM][2 * LEN];
  struct Slot {
    int code;
    double r, i, pf, ar, ai, br, bi;
  };
  // byte offset of the member's n-th step (round rank + team (n / S), step
  // n % S) in an array of doubles: 32 bits beside a scalar base address
  auto at = [&](int n) { return 8u * (uint32_t(((rank + team * (n / S)) * S + n % S) * W) + t); };
  auto get = [](const GMEM double *p, uint32_t o) { return *(const GMEM double *)((const GMEM char *)p + o); };
  auto put = [](GMEM double *p, uint32_t o, double v) { *(GMEM double *)((GMEM char *)p + o) = v; };
  auto load = [&](int n) {
    const uint32_t s = at(n);
    Slot o;
    o.code = *(const GMEM int32_t *)((const GMEM char *)kn + s / 2);
    o.r = get(sumR, s);
    o.i = get(sumI, s);
    o.pf = get(pref, s);
    o.ar = get(dRa, s);
    o.ai = get(dIa, s);
    if constexpr (NM == 2) {
      o.br = get(dRb, s);
      o.bi = get(dIb, s);
    } else {
      o.br = o.bi = 0.0;
      if (pend & 2) {  // the last pass held two moves
        o.br = get(dRb, s);
        o.bi = get(dIb, s);
      }
    }
    return o;
  };
  // the phases of a segment's first k-vector, and of the next along nz
  auto first = [&](int code) {
    const int c0 = code >= 0 ? code : kZeroCode;
#pragma unroll
    for (int v = 0; v < NM; ++v)
#pragma unroll
      for (int p = 0; p < 2 * LEN; ++p) {
        e[v][p] = TablePhase<T>(tab[m0 + v][p], c0);
        // one position (FP32 two) at a time: the scheduler would otherwise
        // hoist every table read and run out of registers
        if (sizeof(T) == 8 || (p & 1)) __builtin_amdgcn_sched_barrier(0);
      }
  };
  auto advance = [&]() {
#pragma unroll
    for (int v = 0; v < NM; ++v)
#pragma unroll
      for (int p = 0; p < 2 * LEN; ++p) {
        e[v][p] = CMul(e[v][p], step[v][p]);
        if (sizeof(T) == 8 && p % 3 == 2) __builtin_amdgcn_sched_barrier(0);
      }
  };
  auto work = [&](int n, const Slot &c) {
    const uint32_t s = at(n);
    const bool used = c.code >= 0;
    double r = (pend & 1) ? c.r + c.ar : c.r, i = (pend & 1) ? c.i + c.ai : c.i;
    r = (pend & 2) ? r + c.br : r;
    i = (pend & 2) ? i + c.bi : i;
    double dR[NM], dI[NM];
#pragma unroll
    for (int v = 0; v < NM; ++v) {
      T sRN = 0, sIN = 0, sRO = 0, sIO = 0;
#pragma unroll
      for (int p = 0; p < LEN; ++p) {
        sRN = Axpy(q[p], e[v][LEN + p].re, sRN);
        sIN = Axpy(q[p], e[v][LEN + p].im, sIN);
        sRO = Axpy(q[p], e[v][p].re, sRO);
        sIO = Axpy(q[p], e[v][p].im, sIO);
      }
      dR[v] = used ? double(sRN - sRO) : 0.0;
      dI[v] = used ? double(sIN - sIO) : 0.0;
    }
    put(sumR, s, r);
    put(sumI, s, i);
    put(dRa, s, dR[0]);
    put(dIa, s, dI[0]);
    e0 += c.pf * (dR[0] * (2.0 * r + dR[0]) + dI[0] * (2.0 * i + dI[0]));
    if constexpr (NM == 2) {
      put(dRb, s, dR[1]);
      put(dIb, s, dI[1]);
      e1 += c.pf * (dR[1] * (2.0 * r + dR[1]) + dI[1] * (2.0 * i + dI[1]));
      const double r1 = r + dR[0], i1 = i + dI[0];
      e2 += c.pf * (dR[1] * (2.0 * r1 + dR[1]) + dI[1] * (2.0 * i1 + dI[1]));
    }
  };
  if (total > 0) {
    Slot x = load(0);
    if constexpr (S == 1) {
#pragma unroll 1
      for (int n = 0; n < total; n += 2) {
        const Slot y = load(min(n + 1, total - 1));
        first(x.code);
        work(n, x);
        x = load(min(n + 2, total - 1));
        if (n + 1 < total) {
          first(y.code);
          work(n + 1, y);
        }
      }
    } else {
#pragma unroll 1
      for (int n0 = 0; n0 < total; n0 += S) {
        first(x.code);
#pragma unroll 1
        for (int j = 0; j < S; j += 2) {
          const Slot y = load(n0 + j + 1);
          if (j > 0) advance();
          work(n0 + j, x);
          x = load(min(n0 + j + 2, total - 1));
          advance();
          work(n0 + j + 1, y);
        }
      }
    }
  }
  const double s0 = WaveSumDpp(e0), s1 = NM == 2 ? WaveSumDpp(e1) : 0.0,
               s2 = NM == 2 ? WaveSumDpp(e2) : 0.0;
  if ((threadIdx.x & (kWave - 1)) == kWave - 1) {
    LMEM double *r = red + (threadIdx.x / kWave) * kXchgVals;
    const bool alone = NM == 1 && m0 == 1;  // B alone: its change from S as it is
    r[kRecA] = alone ? 0.0 : s0;
    r[kRecB0] = alone ? s0 : s1;
    r[kRecB1] = s2;
  }
}

// Adds the pending accepted changes to S(k) at the end of a launch (the
// member's own rounds), in the order the next pass would.
__device__ __noinline__ void RecipFold(const LMEM BatchBox *sb, int rank, int team,
                                       const GMEM int32_t *kn, GMEM double *sumR, GMEM double *sumI,
                                       DeltaPtrs d, int pend) {
  const int per = sb->kSeg * sb->kWidth;  // slots of a round
  for (int r = rank; r < sb->kChunk; r += team)
    for (int s = r * per + int(threadIdx.x); s < (r + 1) * per; s += kBatchThreads) {
      if (kn[s] < 0) continue;
      double re = sumR[s], im = sumI[s];
      if (pend & 1) {
        re += d.R[0][s];
        im += d.I[0][s];
      }
      if (pend & 2) {
        re += d.R[1][s];
        im += d.I[1][s];
      }
      sumR[s] = re;
      sumI[s] = im;
    }
}

// Team exchange, run by wave 0 of each member; lane i < 16 holds value i of
// the member's sums.  Each is published with its 8 lowest mantissa bits
// replaced by the pass tag (seq & 255), so a reader knows a word is this
// pass's without a separate counter: lane i writes word i of the member's 16;
// then lane 16 g + i polls word i of members g, g + 4 until it carries the
// tag.  Slots alternate with the pass's parity, so a stale word is two passes
// old and carries another tag.  Every member clears the tag bits and sums the
// same values in member order (a partial loses at most 2^-44 of itself), so
// all members hold the same bits.  Words go through device-coherent atomics.
// A wait that outlasts kTeamSpinLimit polls sets *err and ok = false.
struct TeamValue {
  double v;
  bool ok;
};

__device__ __forceinline__ uint64_t Tagged(double v, uint64_t tag) {
  return (__builtin_bit_cast(uint64_t, v) & ~uint64_t(0xff)) | tag;
}

__device__ __noinline__ TeamValue TeamSum(GMEM uint64_t *xb, int team, int rank, uint64_t seq,
                                          double v, GMEM int *err) {
  const int lane = int(threadIdx.x) & (kWave - 1), i = lane % kXchgVals, grp = lane / kXchgVals;
  const uint64_t tag = seq & 0xff;
  GMEM uint64_t *data = xb + (seq & 1) * kTeamMax * kXchgVals;
  const uint64_t mine = Tagged(__shfl(v, i), tag);
  if (lane < kXchgVals)
    __hip_atomic_exchange(data + rank * kXchgVals + i, mine, __ATOMIC_RELAXED,
                          __HIP_MEMORY_SCOPE_AGENT);
  uint64_t w[2] = {mine, mine};
  int ok = 1;
  const bool need[2] = {grp < team && grp != rank, grp + 4 < team && grp + 4 != rank};
  for (int64_t n = 0;; ++n) {
    bool all = true;
#pragma unroll
    for (int h = 0; h < 2; ++h)
      if (need[h]) {
        w[h] = __hip_atomic_load(data + (grp + 4 * h) * kXchgVals + i, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
        all = all && (w[h] & 0xff) == tag;
      }
    if (all) break;
    if (n > kTeamSpinLimit) {
      ok = 0;
      break;
    }
  }
  TeamValue out{0.0, __all(ok) != 0};
  if (!out.ok) {
    if (lane == 0) __hip_atomic_exchange(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return out;
  }
  // the tag bits cleared: the partials truncated alike in every member
  const double p0 = __builtin_bit_cast(double, w[0] & ~uint64_t(0xff)),
               p1 = __builtin_bit_cast(double, w[1] & ~uint64_t(0xff));
  for (int m = 0; m < team; ++m) out.v += __shfl(m < 4 ? p0 : p1, (m % 4) * kXchgVals + i);
  return out;
}
static_assert(kXchgVals == 16 && kTeamMax == 8, "four members a wave, twice");

// Bookkeeping of one decided move (Translate/Rotate::Accept,
// src/moves/Translate.h:97-138; MoveSettings::Update,
// src/MoveSettings.cpp:94-146), run by one lane.
__device__ __forceinline__ void Settle(LMEM BatchState *st, bool accept, double lj, double real,
                                       double recip, int type) {
  st->tries[type]++;
  st->tempTries[type]++;
  if (!accept) return;
  st->accepted[type]++;
  st->tempAccepted[type]++;
  st->energy[0] += lj;
  st->energy[2] += real;
  st->energy[3] += recip;
  st->energy[6] = st->energy[0] + st->energy[1] + st->energy[2] + st->energy[3] + st->energy[4] +
                  st->energy[5];
}

// One decision a lane: B after A stayed (lane 1) and after A moved (lane 2) beside A's own (lane
// 0), so a pass waits for one exponential.  Then lane 0 settles the moves.
__device__ __noinline__ void Decide(const LMEM BatchBox *sb, LMEM BatchState *st,
                                    LMEM MoveShared *ms, const LMEM double *uA,
                                    const LMEM double *uB, int has, const LMEM BatchTrace *trace,
                                    int64_t at) {
  const int lane = int(threadIdx.x) & (kWave - 1);
  const LMEM double *s = ms->tot;
  const int x = lane == 2 ? 3 : 0;  // kX...1 after kX...0
  double lj, real, recip, ov;
  if (lane == 0) {
    lj = s[kLjA];
    real = s[kRealA];
    recip = s[kRecA];
    ov = s[kOvA];
  } else {
    lj = s[kLjB] + s[kXLj0 + x];
    real = s[kRealB] + s[kXReal0 + x];
    recip = lane == 2 ? s[kRecB1] : s[kRecB0];
    ov = s[kOvB] + s[kXOv0 + x];
  }
  const double dE = lj + real + recip;
  const bool res = (lane == 0 ? uA[5] : uB[5]) < exp(-sb->beta * dE) && !(ov > 0.0);
  const uint64_t yes = __ballot(res);
  const bool accA = (has & 1) && (yes & 1);
  const bool accB = (has & 2) && ((yes >> (accA ? 2 : 1)) & 1);
  // the deciding lanes keep their terms; lane 0 reads B's
  const int lb = accA ? 2 : 1;
  const double ljB = __shfl(lj, lb), realB = __shfl(real, lb), recipB = __shfl(recip, lb),
               ovB = __shfl(ov, lb);
  if (lane != 0) return;
  if (has & 1) Settle(st, accA, lj, real, recip, ms->mv[0].type);
  if (has & 2) Settle(st, accB, ljB, realB, recipB, ms->mv[1].type);
  ms->accept[0] = accA;
  ms->accept[1] = accB;
  if (trace) {
    if ((has & 1) && at < trace->cap) {
      trace->acc[at] = accA;
      trace->dlj[at] = lj;
      trace->dreal[at] = real;
      trace->drecip[at] = ov > 0.0 ? 0.0 : recip;
    }
    const int64_t b = at + (has == 3 ? 1 : 0);
    if ((has & 2) && b < trace->cap) {
      trace->acc[b] = accB;
      trace->dlj[b] = ljB;
      trace->dreal[b] = realB;
      trace->drecip[b] = ovB > 0.0 ? 0.0 : recipB;
    }
  }
}

// ------------------------------------------------------------- programs --
// The pair waves and the reciprocal waves of a workgroup run a program each,
// a loop over the box's passes with the same four barriers a pass (five where
// draws are made): called once a box, so the callee-saved registers of the
// phases (60 stores a lane in FP64) are saved once, not once a pass, which holds
// 7 spill stores and 18 loads of its own and the small frames of the
// out-of-line steps.  Which moves a pass holds follows from the draws and
// the step alone, so every wave finds it for itself.
// A run's pointers lie in LDS, one copy a workgroup: in a lane's private memory
// they were 300 bytes of scratch stored by each of 1024 lanes, and the trace's
// address took the kernel's arguments there too, 21 us of every launch.
template <typename T>
struct BoxRun {
  const LMEM BatchBox *sb;
  LMEM BatchState *st;
  LMEM MoveShared *ms;
  LMEM PhaseTab<T> *tab;
  LMEM CoulTab *ctab;
  LMEM PairQueue *queues;
  LMEM int *nearList;
  LMEM double (*draws)[8];
  LMEM float *CX, *CY, *CZ;  // centres in LDS (null: not there)
  GMEM double *X, *Y, *Z, *CXg, *CYg, *CZg;
  const GMEM int32_t *kn;
  const GMEM double *pref;
  GMEM double *sumR, *sumI;
  DeltaPtrs delta;
  GMEM uint64_t *xb;
  GMEM int *err;
  BatchTrace trace;
  int64_t step, end;
  uint64_t pass;
  int rank, team, pairs;    // pairs: passes of two moves
  int traced;               // 1: this member writes the trace
};

// Where a box's run stands, the same in every wave.  An even step A and the
// odd step B after it go together if both are in the launch, move different
// molecules and no adjustment of the move settings falls before either (B's
// proposal would need A's outcome).
struct Cursor {
  int64_t step, end, drawn;  // drawn: first step of the draws in LDS
  uint64_t pass;
  int pend;                  // moves of the last pass accepted, their change of S(k) pending
  int has, skip;             // moves of this pass (bit 0 A, bit 1 B); A's molecule for CrossTerms
  int uA, uB;                // their draws
  bool adjust;
};

template <typename T>
__device__ __forceinline__ Cursor Begin(const BoxRun<T> &r) {
  return Cursor{UniformI64(r.step), UniformI64(r.end), -1, uint64_t(UniformI64(int64_t(r.pass))),
                0, 0, -1, 0, 0, false};
}

// The next pass; draws are made kDrawChunk steps at a time from an even one.
template <typename T>
__device__ __forceinline__ void NextPass(const BoxRun<T> &r, Cursor &c, int nmols,
                                         int64_t perAdjust) {
  const int64_t even = c.step & ~int64_t(1);
  if (c.drawn < 0 || even + 1 >= c.drawn + kDrawChunk) {
    c.drawn = even;
    if (threadIdx.x < kDrawChunk)
      MoveDraws(r.sb->seed, uint64_t(c.drawn + threadIdx.x), r.draws[threadIdx.x]);
    __syncthreads();
  }
  c.uA = int(even - c.drawn);
  c.uB = c.uA + 1;
  const int molA = __builtin_amdgcn_readfirstlane(PickMol(r.draws[c.uA][1], nmols));
  const int molB = __builtin_amdgcn_readfirstlane(PickMol(r.draws[c.uB][1], nmols));
  c.adjust = uint64_t(c.step + 1) % uint64_t(perAdjust) == 0;
  c.has = 2;
  if (c.step == even)
    c.has = (r.pairs && c.step + 1 < c.end && molA != molB && !c.adjust &&
             uint64_t(c.step + 2) % uint64_t(perAdjust) != 0)
                ? 3
                : 1;
  c.skip = (c.has & 2) && molA != molB ? molA : -1;
}

// After a pass's last barrier; false: a team exchange failed.
template <typename T>
__device__ __forceinline__ bool EndPass(const BoxRun<T> &r, Cursor &c) {
  if (__builtin_amdgcn_readfirstlane(r.ms->abort)) return false;
  const int accA = __builtin_amdgcn_readfirstlane(r.ms->accept[0]),
            accB = __builtin_amdgcn_readfirstlane(r.ms->accept[1]);
  // a move alone keeps its change in the first arrays
  c.pend = c.has == 3 ? (accA | (accB << 1)) : (c.has == 1 ? accA : accB);
  c.step += c.has == 3 ? 2 : 1;
  ++c.pass;
  return true;
}

__device__ __forceinline__ void WaveFence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Totals, decisions and commit of a pass, by wave 0.
template <typename T>
__device__ __noinline__ void FinishPass(const LMEM BoxRun<T> *r, int uA, int uB, int has, uint64_t pass,
                                        int64_t at, int pw, int waves, int len) {
  LMEM MoveShared *ms = r->ms;
  const LMEM double *red = &ms->red[0][0];
  const int tid = threadIdx.x, i = tid % kXchgVals;
  // value i comes from the pair waves, the reciprocal waves or the last pair wave
  const int w0 = i < kRecA ? 0 : (i < kXLj0 ? pw : pw - 1);
  const int w1 = i < kRecA ? pw : (i < kXLj0 ? waves : (r->rank == 0 ? pw : pw - 1));
  double v = 0.0;
  for (int w = w0; w < w1; ++w) v += red[w * kXchgVals + i];
  if (i >= kNumSums) v = 0.0;
  if (r->team > 1) {
    const TeamValue t = TeamSum(r->xb, r->team, r->rank, pass + 1, v, r->err);
    v = t.v;
    if (!t.ok) {
      if (tid == 0) ms->abort = 1;
      return;
    }
  }
  if (tid < kXchgVals) ms->tot[tid] = v;
  WaveFence();
  Decide(r->sb, r->st, ms, r->draws[uA], r->draws[uB], has, r->traced ? &r->trace : nullptr, at);
  WaveFence();
  // S(k) follows in the next pass's reciprocal phase
  const int mvI = tid / 32, p = tid % 32;
  const LMEM MoveOne *mv = &ms->mv[mvI];
  if (((has >> mvI) & 1) && ms->accept[mvI]) {
    const int m = mv->mol;
    if (p < len) {
      const int64_t ai = int64_t(m) * len + p;
      r->X[ai] = mv->newp[0][p];
      r->Y[ai] = mv->newp[1][p];
      r->Z[ai] = mv->newp[2][p];
    }
    if (p == 0 && mv->type == 0) {
      r->CXg[m] = mv->com[1][0];
      r->CYg[m] = mv->com[1][1];
      r->CZg[m] = mv->com[1][2];
      if (r->CX) {
        r->CX[m] = float(mv->com[1][0]);
        r->CY[m] = float(mv->com[1][1]);
        r->CZ[m] = float(mv->com[1][2]);
      }
    }
  }
}

// The pair waves' program; wave 0 also proposes, decides and commits.
template <typename T, int LEN, typename ComPtr>
__device__ __noinline__ Cursor PairProgram(const LMEM BoxRun<T> *rp, ComPtr CX, ComPtr CY, ComPtr CZ) {
  BoxRun<T> r = *(const BoxRun<T> *)rp;
  r.X = UniformPtr(r.X);
  r.Y = UniformPtr(r.Y);
  r.Z = UniformPtr(r.Z);
  r.rank = __builtin_amdgcn_readfirstlane(r.rank);
  r.team = __builtin_amdgcn_readfirstlane(r.team);
  const LMEM BatchBox *sb = r.sb;
  LMEM MoveShared *ms = r.ms;
  LMEM double *red = &ms->red[0][0];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int pw = __builtin_amdgcn_readfirstlane(sb->pairWaves);
  const int nmols = __builtin_amdgcn_readfirstlane(sb->nmols);
  const bool ewald = __builtin_amdgcn_readfirstlane(sb->ewald) != 0;
  const int64_t perAdjust = UniformI64(sb->perAdjust);
  Cursor c = Begin(r);
  const int64_t start = c.step;
  while (c.step < c.end) {
    NextPass(r, c, nmols, perAdjust);
    if (wave == 0) {  // proposals and trial coordinates, lanes 32 up for B
      const int tid = threadIdx.x;
      if (c.adjust) {
        if (tid == 0) Adjust(sb, r.st);
        WaveFence();
      }
      const int v = tid / 32, p = tid % 32;
      if (p < LEN && ((c.has >> v) & 1))
        Propose(sb, r.st, &ms->mv[v], r.draws[v ? c.uB : c.uA], p, r.X, r.Y, r.Z, r.CXg, r.CYg, r.CZg);
    }
    __syncthreads();
    if (ewald) BuildTables<T>(sb, ms->mv, LEN, c.has == 2 ? 1 : 0, c.has == 3 ? 2 : 1, r.tab);
    __syncthreads();  // tables complete
    PairPhase<T, LEN>(sb, r.ctab, ms->mv, r.X, r.Y, r.Z, CX, CY, CZ, nmols, r.rank, r.team, c.has,
                      c.skip, r.queues, r.nearList, red);
    if (wave == pw - 1 && r.rank == 0)
      CrossTerms<T>(sb, r.ctab, ms->mv, r.X, r.Y, r.Z, LEN, c.has, c.skip, red + wave * kXchgVals);
    __syncthreads();
    if (wave == 0)
      FinishPass<T>(rp, c.uA, c.uB, c.has, c.pass, c.step - start, pw,
                    ewald ? kBatchThreads / kWave : pw, LEN);
    __syncthreads();
    if (!EndPass(r, c)) break;
  }
  return c;
}

// The reciprocal waves' program.
template <typename T, int S, int LEN>
__device__ __noinline__ Cursor RecipProgram(const LMEM BoxRun<T> *rp) {
  const BoxRun<T> r = *(const BoxRun<T> *)rp;
  const LMEM BatchBox *sb = r.sb;
  LMEM double *red = &r.ms->red[0][0];
  const int nmols = __builtin_amdgcn_readfirstlane(sb->nmols);
  const bool ewald = __builtin_amdgcn_readfirstlane(sb->ewald) != 0;
  const int64_t perAdjust = UniformI64(sb->perAdjust);
  Cursor c = Begin(r);
  while (c.step < c.end) {
    NextPass(r, c, nmols, perAdjust);
    __syncthreads();
    if (ewald) BuildTables<T>(sb, r.ms->mv, LEN, c.has == 2 ? 1 : 0, c.has == 3 ? 2 : 1, r.tab);
    __syncthreads();  // tables complete
    if (ewald) {
      if (c.has == 3)
        RecipPhase<T, S, LEN, 2>(sb, r.tab, 0, r.kn, r.pref, r.sumR, r.sumI, r.delta, r.rank, r.team,
                                 c.pend, red);
      else
        RecipPhase<T, S, LEN, 1>(sb, r.tab, c.has == 2 ? 1 : 0, r.kn, r.pref, r.sumR, r.sumI, r.delta,
                                 r.rank, r.team, c.pend, red);
    }
    __syncthreads();
    __syncthreads();
    if (!EndPass(r, c)) break;
  }
  return c;
}

template <typename T, int LEN>
__device__ __forceinline__ Cursor RunBox(const LMEM BoxRun<T> *r, int wave) {
  if (wave < __builtin_amdgcn_readfirstlane(r->sb->pairWaves)) {
    if (r->CX) return PairProgram<T, LEN>(r, r->CX, r->CY, r->CZ);
    return PairProgram<T, LEN>(r, r->CXg, r->CYg, r->CZg);
  }
  switch (__builtin_amdgcn_readfirstlane(r->sb->kSeg)) {
    case 8:
      return RecipProgram<T, 8, LEN>(r);
    case 4:
      return RecipProgram<T, 4, LEN>(r);
    case 2:
      return RecipProgram<T, 2, LEN>(r);
    default:
      return RecipProgram<T, 1, LEN>(r);
  }
}

template <int PREC>
__global__ void __launch_bounds__(kBatchThreads) McBatchKernel(const BatchArgs a) {
  using T = typename Prec<PREC>::T;
  __shared__ BatchBox sbS;
  __shared__ double drawsS[kDrawChunk][8];
  __shared__ PhaseTab<T> tabS[2];
  __shared__ MoveShared msS;
  __shared__ BatchState stS;  // running energies and move settings
  __shared__ PairQueue queuesS[kPairWavesMax];
  __shared__ int nearListS[kPairWavesMax * 2 * kNearListLen];
  __shared__ CoulTab ctabS;
  __shared__ BoxRun<T> runS;
  extern __shared__ float ldsCom[];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  for (int ti = a.wgTask[blockIdx.x]; ti < a.wgTask[blockIdx.x + 1]; ++ti) {
    const BatchTask task = a.tasks[ti];
    const int b = __builtin_amdgcn_readfirstlane(task.box);
    const int rank = __builtin_amdgcn_readfirstlane(task.rank);
    {
      const uint64_t *src = reinterpret_cast<const uint64_t *>(&a.boxes[b]);
      uint64_t *dst = reinterpret_cast<uint64_t *>(&sbS);
      // the Coulomb table's loads run beside the description's
      constexpr int kPer = (kTabWords / 2 + kBatchThreads - 1) / kBatchThreads;
      TabPair row[kPer];
      if (PREC == 0) {
        const GMEM TabPair *t = (const GMEM TabPair *)(a.coulTab + size_t(a.boxes[b].tab) * kTabWords);
#pragma unroll
        for (int i = 0; i < kPer; ++i) row[i] = t[min(tid + i * kBatchThreads, kTabWords / 2 - 1)];
      }
      for (int i = tid; i < int(sizeof(BatchBox) / 8); i += kBatchThreads) dst[i] = src[i];
      if (PREC == 0) {
#pragma unroll
        for (int i = 0; i < kPer; ++i)
          if (tid + i * kBatchThreads < kTabWords / 2)
            ((LMEM TabPair *)Lp(ctabS.c))[tid + i * kBatchThreads] = row[i];
      }
    }
    if (tid == 0) {
      msS.abort = 0;
      stS = a.state[b];
    }
    if (tid == kWave) {
      const BatchBox &box = a.boxes[b];
      const int64_t aoff = box.atomOff, moff = box.molOff, koff = box.kOff;
      BoxRun<T> &r = runS;
      r.sb = Lp(&sbS);
      r.st = Lp(&stS);
      r.ms = Lp(&msS);
      r.tab = Lp(tabS);
      r.ctab = Lp(&ctabS);
      r.queues = Lp(queuesS);
      r.nearList = Lp(nearListS);
      r.draws = Lp(drawsS);
      // The box's molecule centres, rounded to FP32, live in LDS for the launch
      // when they fit (a.ldsMols per workgroup): the cull reads them there.
      r.CX = box.nmols <= a.ldsMols ? Lp(ldsCom) : nullptr;
      r.CY = r.CX + a.ldsMols;
      r.CZ = r.CX + 2 * a.ldsMols;
      // Team members share the box's coordinates and centres.  Every member
      // writes the same accepted values at the same point of a pass, after the
      // exchange that needs all members' pair phases of that pass, and reads
      // them only after its own write and a barrier: a read sees its own
      // member's write or another's identical one.
      r.X = Gp(a.x + aoff);
      r.Y = Gp(a.y + aoff);
      r.Z = Gp(a.z + aoff);
      r.CXg = Gp(a.cx + moff);
      r.CYg = Gp(a.cy + moff);
      r.CZg = Gp(a.cz + moff);
      r.kn = Gp(a.kn + koff);
      r.pref = Gp(a.pref + koff);
      r.sumR = Gp(a.sumR + koff);
      r.sumI = Gp(a.sumI + koff);
      r.delta = DeltaPtrs{{Gp(a.dR + koff), Gp(a.dR2 ? a.dR2 + koff : a.dR + koff)},
                          {Gp(a.dI + koff), Gp(a.dI2 ? a.dI2 + koff : a.dI + koff)}};
      r.xb = Gp(a.xchg + int64_t(b) * kXchgWords);
      r.err = Gp(a.err);
      r.trace = a.trace;
      r.traced = rank == 0 && b == a.trace.box;
      r.step = a.state[b].step;
      r.end = r.step + a.moves[b];
      r.pass = uint64_t(a.state[b].passes);
      r.rank = rank;
      r.team = box.team > 1 ? box.team : 1;
      r.pairs = a.dR2 != nullptr;
    }
    __syncthreads();
    const LMEM BatchBox *sb = Lp(&sbS);
    const LMEM BoxRun<T> *r = Lp(&runS);
    const int len = __builtin_amdgcn_readfirstlane(sb->molLen);
    const int nmols = __builtin_amdgcn_readfirstlane(sb->nmols);
    const int64_t moves = UniformI64(r->end - r->step);
    const bool ewald = __builtin_amdgcn_readfirstlane(sb->ewald) != 0;
    const bool inLds = nmols <= a.ldsMols;
    const uint64_t t0 = wall_clock64();
    if (moves > 0) {
      if (inLds)
        for (int i = tid; i < nmols; i += kBatchThreads) {
          Lp(ldsCom)[i] = float(r->CXg[i]);
          Lp(ldsCom)[a.ldsMols + i] = float(r->CYg[i]);
          Lp(ldsCom)[2 * a.ldsMols + i] = float(r->CZg[i]);
        }
      // the centres are read after the programs' first barrier
      Cursor c;
      switch (len) {
        case 1:
          c = RunBox<T, 1>(r, wave);
          break;
        case 2:
          c = RunBox<T, 2>(r, wave);
          break;
        case 3:
          c = RunBox<T, 3>(r, wave);
          break;
        default:
          c = RunBox<T, 4>(r, wave);
      }
      if (c.pend && ewald) {
        const BoxRun<T> &g = runS;
        RecipFold(sb, rank, g.team, g.kn, g.sumR, g.sumI, g.delta, c.pend);
      }
      if (tid == 0 && rank == 0) {
        stS.step = c.step;
        stS.passes = int64_t(c.pass);
        a.state[b] = stS;
      }
    }
    if (tid == 0 && rank == 0) a.boxTicks[b] = wall_clock64() - t0;
    __syncthreads();  // LDS is reused by the next task
  }
}

}  // namespace

template <int PREC>
static hipError_t SetLds(int ldsMols) {
  const size_t dyn = sizeof(float) * 3 * size_t(ldsMols);
  return hipFuncSetAttribute(reinterpret_cast<const void *>(&McBatchKernel<PREC>),
                             hipFuncAttributeMaxDynamicSharedMemorySize, int(dyn));
}

template <int PREC>
static hipError_t LaunchOne(int grid, const BatchArgs &a, hipStream_t s, bool setAttr) {
  const size_t dyn = sizeof(float) * 3 * size_t(a.ldsMols);
  if (setAttr) {
    hipError_t e = SetLds<PREC>(a.ldsMols);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(McBatchKernel<PREC>, dim3(grid), dim3(kBatchThreads), dyn, s, a);
  return hipGetLastError();
}

template <int PREC>
static hipError_t ResidentOne(int ldsMols, int *perCU) {
  hipError_t e = SetLds<PREC>(ldsMols);
  if (e != hipSuccess) return e;
  const size_t dyn = sizeof(float) * 3 * size_t(ldsMols);
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(perCU, McBatchKernel<PREC>, kBatchThreads,
                                                      dyn);
}

hipError_t BatchResidentPerCU(int precision, int ldsMols, int *perCU) {
  return precision == 1 ? ResidentOne<1>(ldsMols, perCU) : ResidentOne<0>(ldsMols, perCU);
}

hipError_t PrepareBatch(int precision, int ldsMols) {
  return precision == 1 ? SetLds<1>(ldsMols) : SetLds<0>(ldsMols);
}

int BatchLdsMols(int maxMols) { return maxMols < kBatchLdsMolCap ? maxMols : kBatchLdsMolCap; }

hipError_t LaunchBatch(int precision, int grid, const BatchArgs &a, hipStream_t s, bool setAttr) {
  return precision == 1 ? LaunchOne<1>(grid, a, s, setAttr) : LaunchOne<0>(grid, a, s, setAttr);
}

}  // namespace gomc
