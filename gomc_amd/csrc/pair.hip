// Whole-box pair sums on the plain path: the real-space energy of a box
// (CalculateEnergy::BoxInter, src/CalculateEnergy.cpp:157-266), the pair
// forces of MultiParticle moves (BoxForce, 268-406) and the pair virial
// (VirialCalc, 411-579).
//
// Molecules, not atoms, are put in cells and tested first: two molecules
// whose centres are farther apart than the cutoff plus both radii hold no
// pair inside it (triangle inequality on minimum-image distances), and the
// test covers all their atom pairs at once.  In water at rc = 12 A the
// 27-cell neighbourhood of an atom list has 9 pairs outside the cutoff for
// each one inside; of the atom pairs of near molecules 63 % are inside, so
// they are evaluated as they come, 64 at a time, without a list of the ones
// that count.
//
// One wave (S waves in a small box) owns a home molecule.  It walks the
// molecules of the cells around it, 16 lanes to a run of cells consecutive
// in z, appends the atoms of near ones to a list in its LDS and, whenever
// the list holds 64, takes them one per lane against each home atom.
// Forces: every pair is met from both ends and the sums of a home atom stay
// in registers until the end, so there are no atomics and the order of
// every sum is fixed by the positions.  Energies and virials: the partner
// must come later in the cell order, so each pair is met once.
//
// Bound by FP64 issue and the tail of the last round of home molecules (128
// VGPRs, four waves a SIMD, of which three are there on average).
// 10,000 waters, rc 12 A: forces 333 us (with atom cells, tiles and sorted
// hit lists 733), virial 166 us (606), energy 185 us (950); 1000 waters, rc
// 10 A: forces 62 us (154).
#include <algorithm>
#include <cmath>

#include "box.hpp"

namespace gomc {
namespace {

constexpr int kPairThreads = 256, kPairWaves = kPairThreads / kWave;
constexpr int kHomeAtoms = 4;  // home atoms per pass; a longer molecule makes several
constexpr int kAtomList = kWave - 1 + kWave * kMaxMolAtoms;
constexpr int kPairTypesLds = 8;  // atom types whose pair table fits in LDS

// ------------------------------------------------------- molecules by cell --
struct MolCellArgs {
  BoxGeom g;
  const double *x, *y, *z;
  const int *mol, *molStart;
  int nmols, ncell, n[3];
  double cs[3];
  int *count, *start;      // [ncell], [ncell + 1]; count is zero between builds
  int *cell, *slot, *tmp;  // [nmols]
  double4 *where, *pack;   // [nmols] centre and radius, by molecule and sorted
  int *sid;                // [nmols] molecule of each sorted place
  unsigned long long *radBits;  // [2] largest radius: being gathered, of the last build
};

// Centre (mean of the atoms, each by its minimum image from the first) and
// radius of every molecule in the box, and its place in its cell.
__global__ void __launch_bounds__(kBlock) MolPlaceKernel(const MolCellArgs a) {
  const int m = blockIdx.x * kBlock + threadIdx.x;
  if (m >= a.nmols) return;
  const int s = a.molStart[m], e = a.molStart[m + 1];
  if (a.mol[s] < 0) {
    a.cell[m] = -1;
    return;
  }
  const double x0 = a.x[s], y0 = a.y[s], z0 = a.z[s];
  double sx = 0.0, sy = 0.0, sz = 0.0;
  for (int p = s + 1; p < e; ++p) {
    sx += MinImage(a.x[p] - x0, a.g.L[0], a.g.half[0]);
    sy += MinImage(a.y[p] - y0, a.g.L[1], a.g.half[1]);
    sz += MinImage(a.z[p] - z0, a.g.L[2], a.g.half[2]);
  }
  const double inv = 1.0 / double(e - s);
  sx *= inv;
  sy *= inv;
  sz *= inv;
  double r2 = sx * sx + sy * sy + sz * sz;
  for (int p = s + 1; p < e; ++p) {
    const double dx = MinImage(a.x[p] - x0, a.g.L[0], a.g.half[0]) - sx;
    const double dy = MinImage(a.y[p] - y0, a.g.L[1], a.g.half[1]) - sy;
    const double dz = MinImage(a.z[p] - z0, a.g.L[2], a.g.half[2]) - sz;
    r2 = fmax(r2, dx * dx + dy * dy + dz * dz);
  }
  const double rad = sqrt(r2);
  const double cx = Wrap(x0 + sx, a.g.L[0]), cy = Wrap(y0 + sy, a.g.L[1]), cz = Wrap(z0 + sz, a.g.L[2]);
  const int c = CellOf(cx, cy, cz, a.cs, a.n);
  a.where[m] = make_double4(cx, cy, cz, rad);
  a.cell[m] = c;
  a.slot[m] = atomicAdd(&a.count[c], 1);
  // positive doubles order as their bits do
  atomicMax(&a.radBits[0], (unsigned long long)__builtin_bit_cast(uint64_t, rad));
}

// Exclusive scan of the counts (one workgroup), which are cleared for the
// next build; the largest radius moves to its place.
__global__ void __launch_bounds__(1024) MolScanKernel(const MolCellArgs a) {
  __shared__ int waveSum[16];
  const int t = threadIdx.x, lane = t % kWave, w = t / kWave;
  if (t == 0) {
    a.radBits[1] = a.radBits[0];
    a.radBits[0] = 0;
  }
  int run = 0;
  for (int c0 = 0; c0 < a.ncell; c0 += 1024) {
    const int c = c0 + t, n = c < a.ncell ? a.count[c] : 0;
    int incl = n;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      const int u = __shfl_up(incl, d);
      if (lane >= d) incl += u;
    }
    if (lane == kWave - 1) waveSum[w] = incl;
    __syncthreads();
    int before = run, all = 0;
    for (int i = 0; i < 16; ++i) {
      if (i < w) before += waveSum[i];
      all += waveSum[i];
    }
    if (c < a.ncell) {
      a.start[c] = before + incl - n;
      a.count[c] = 0;
    }
    run += all;
    __syncthreads();
  }
  if (t == 0) a.start[a.ncell] = run;
}

__global__ void __launch_bounds__(kBlock) MolScatterKernel(const MolCellArgs a) {
  const int m = blockIdx.x * kBlock + threadIdx.x;
  if (m < a.nmols && a.cell[m] >= 0) a.tmp[a.start[a.cell[m]] + a.slot[m]] = m;
}

// Each cell in ascending molecule order, whatever order the atomics gave.
__global__ void __launch_bounds__(kBlock) MolSortKernel(const MolCellArgs a) {
  const int m = blockIdx.x * kBlock + threadIdx.x;
  if (m >= a.nmols || a.cell[m] < 0) return;
  const int s = a.start[a.cell[m]], e = a.start[a.cell[m] + 1];
  int rank = 0;
  for (int i = s; i < e; ++i) rank += a.tmp[i] < m;
  a.pack[s + rank] = a.where[m];
  a.sid[s + rank] = m;
}

// -------------------------------------------------------------- pair sums --
enum : int { kEnergy = 0, kForce = 1, kVirial = 2 };

struct PairArgs {
  BoxGeom g;
  double invL[3], rCut;
  const double *x, *y, *z, *q;
  const int *type, *molStart;
  const double *sigSq, *epsCn, *nHalf, *epsCn6, *nOver6;
  int ntypes, nmols;
  int uniLen;  // atoms of every molecule, 0 if they differ
  int ncell, n[3];
  double cs[3];
  const int *start, *sid;
  const double4 *pack;
  const unsigned long long *radBits;
  double *fx, *fy, *fz;        // kForce
  const double *cx, *cy, *cz;  // kVirial: molecule centres as the driver keeps them
  const int *mol;
  double *vpart;               // kVirial: [blocks][6]
  Partial4 *partials;          // kEnergy, kForce
  unsigned *counter;
  double *result;
};

struct PairType {
  double sig, eps, nh, eps6, nov6;
};

// The cells to visit along one axis: `cnt` cells from `first` (periodic).
struct CellRange {
  int first, cnt;
};
__device__ __forceinline__ CellRange Range(int at, int n, int reach) {
  return 2 * reach + 1 >= n ? CellRange{0, n} : CellRange{at - reach, 2 * reach + 1};
}

struct PairTerms {
  double eLJ, eReal, vLJ, vReal;
};

// Energies and virial factors F.r / r^2 of one pair inside the box cutoff
// (FFParticle::CalcCoulomb / CalcCoulombVir, src/FFParticle.cpp:387-446,
// CalcEn / CalcVir 295-359): one reciprocal square root (a Newton-refined
// estimate, then corrections for r, sigma^2 / r^2 and 1 / r^2, to the last place)
// stands for every root and division, and one exponential for erfc's and the
// virial's Gaussian.  The energy alone takes libm's erfc and pow: the
// polynomial is 4e-16 too small in the mean, which a sum over all pairs keeps
// (Coulomb energy of 300 to 2197 waters within 3e-16 of 64-bit sums, by the
// polynomial within 4e-15).
template <bool E, bool F, bool MIE>  // MIE: some repulsion exponent is not 12
__device__ __forceinline__ PairTerms PairEval(const BoxGeom &g, Coefs c, double d2, double qiqj,
                                              const PairType &t) {
  constexpr bool libm = E && !F;
  PairTerms p{0.0, 0.0, 0.0, 0.0};
  d2 = fmax(d2, 0x1p-1022);  // coincident atoms: huge, not 0 x inf
  const double ir = Rsqrt64(d2);
  double ir2 = ir * ir;
  if (F) ir2 = fma(ir2, fma(-d2, ir2, 1.0), ir2);
  if (g.elect && qiqj != 0.0 && !(g.rCutCoulSq < d2)) {
    if (g.ewald) {
      double dist = d2 * ir;
      dist = fma(fma(-dist, dist, d2), 0.5 * ir, dist);
      const double x = g.alpha * dist;
      if (libm) {
        p.eReal = qiqj * (erfc(x) * ir);
      } else {
        const double gauss = ExpNeg(c, -(x * x));
        double ex;
        if (x <= kErfcxUse) {
          const double u = (x - kErfcxMid) * kErfcxInvHalf;
          ex = c[kExpDeg + 1];
#pragma unroll
          for (int k = 1; k <= kErfcxDeg; ++k) ex = FmaS(ex, u, c[kExpDeg + 1 + k]);
        } else {
          ex = ErfcxTail(x);
        }
        const double ec = gauss * ex * ir;
        if (E) p.eReal = qiqj * ec;
        p.vReal = qiqj * (ec + g.alpha * M_2_SQRTPI * gauss) * ir2;
      }
    } else {
      if (E) p.eReal = qiqj * ir;
      if (F) p.vReal = qiqj * (ir2 * ir);
    }
  }
  if (t.eps6 != 0.0 && !(g.rCutLJSq < d2)) {
    const double rRat2 = E ? LJRatio(t.sig, d2, ir) : t.sig * ir2;
    const double att = rRat2 * rRat2 * rRat2;
    double rep = att * att;
    if (MIE && t.nh != 6.0) rep = libm ? pow(rRat2, t.nh) : MiePow(rRat2, t.nh);
    if (E) p.eLJ = t.eps * (rep - att);
    if (F) p.vLJ = t.eps6 * (t.nov6 * rep - att) * ir2;
  }
  return p;
}

__device__ __forceinline__ void WaveSync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

struct HomeAtom {
  double x, y, z, q;
};

template <int MODE, int S, bool MIE>
__global__ void __launch_bounds__(kPairThreads, MIE ? 2 : 4) PairKernel(const PairArgs a) {
  constexpr bool kE = MODE != kVirial, kF = MODE != kEnergy;
  __shared__ int lists[kPairWaves][kAtomList];
  __shared__ HomeAtom homes[kPairWaves][kHomeAtoms];
  __shared__ int htype[kPairWaves][kHomeAtoms];
  __shared__ double tab[5][kPairTypesLds * kPairTypesLds];
  __shared__ double red[kPairWaves][3 * kHomeAtoms];
  __shared__ double bred[kPairWaves];
  const int tid = threadIdx.x, lane = tid % kWave;
  const int w = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int nt2 = a.ntypes * a.ntypes;
  const bool inLds = a.ntypes <= kPairTypesLds;
  if (inLds)
    for (int i = tid; i < nt2; i += kPairThreads) {
      tab[0][i] = a.sigSq[i];
      tab[1][i] = a.epsCn[i];
      tab[2][i] = a.nHalf[i];
      tab[3][i] = a.epsCn6[i];
      tab[4][i] = a.nOver6[i];
    }
  __syncthreads();
  const int u = blockIdx.x * (kPairWaves / S) + w / S;  // home's place in the cell order
  const int slice = w % S;
  const bool on = u < a.start[a.ncell];
  int *list = lists[w];
  const Coefs coefs = GetCoefs();
  double lj = 0.0, real = 0.0;            // energies
  double v[6] = {0, 0, 0, 0, 0, 0};       // virial: LJ xx yy zz, real xx yy zz
  int a0 = 0, len = 0;
  if (on) {
    const int m = __builtin_amdgcn_readfirstlane(a.sid[u]);
    a0 = a.molStart[m];
    len = a.molStart[m + 1] - a0;
    const double4 home = a.pack[u];
    const double near = a.rCut + 1e-6 + home.w;
    const double widest = a.rCut + 1e-6 +
        2.0 * __builtin_bit_cast(double, uint64_t(a.radBits[1]));
    const int c = CellOf(home.x, home.y, home.z, a.cs, a.n);
    const CellRange rx = Range(c / (a.n[1] * a.n[2]), a.n[0], int(ceil(widest / a.cs[0]))),
                    ry = Range((c / a.n[2]) % a.n[1], a.n[1], int(ceil(widest / a.cs[1]))),
                    rz = Range(c % a.n[2], a.n[2], int(ceil(widest / a.cs[2])));
    // the range of z as one run of cells, or two where it wraps
    const int zA = rz.first < 0 ? rz.first + a.n[2] : rz.first;
    const int nA = min(rz.cnt, a.n[2] - zA), nB = rz.cnt - nA;
    const int cols = rx.cnt * ry.cnt, runs = nB > 0 ? 2 * cols : cols;
    double hcx = 0, hcy = 0, hcz = 0;
    if (MODE == kVirial) {
      hcx = a.cx[m];
      hcy = a.cy[m];
      hcz = a.cz[m];
    }
    for (int h0 = 0; h0 < len; h0 += kHomeAtoms) {
      const int nh = min(kHomeAtoms, len - h0);
      WaveSync();
      if (lane < nh) {
        const int i = a0 + h0 + lane;
        homes[w][lane] = HomeAtom{a.x[i], a.y[i], a.z[i], a.q[i]};
        int lj = a.ntypes > kWave;
        for (int t = 0; t < min(a.ntypes, kWave); ++t)
          lj |= a.epsCn6[a.type[i] + t * a.ntypes] != 0.0;
        htype[w][lane] = a.type[i] | (lj << 30);  // bit 30: some type interacts by LJ with it
      }
      WaveSync();
      double f[kHomeAtoms][3] = {};
      int count = 0;  // atoms listed, wave-uniform
      int r0 = slice * 4 - 4 * S, at = 0, end = 0;
      bool more = true;
      for (;;) {
        // cull until a batch is full
        while (count < kWave && more) {
          if (!__any(at < end)) {
            r0 += 4 * S;
            if (r0 >= runs) {
              more = false;
              break;
            }
            const int r = r0 + lane / 16;
            at = end = 0;
            if (r < runs) {
              const int col = r < cols ? r : r - cols;
              int ix = rx.first + col / ry.cnt, iy = ry.first + col % ry.cnt;
              ix += ix < 0 ? a.n[0] : (ix >= a.n[0] ? -a.n[0] : 0);
              iy += iy < 0 ? a.n[1] : (iy >= a.n[1] ? -a.n[1] : 0);
              const int base = (ix * a.n[1] + iy) * a.n[2];
              const int lo = base + (r < cols ? zA : 0), hi = lo + (r < cols ? nA : nB);
              at = a.start[lo];
              end = a.start[hi];
              if (MODE != kForce) at += max(0, (u + 1 - at) / 16 * 16);  // places before u
              at += lane % 16;
            }
            continue;
          }
          bool hit = false;
          int first = 0, n = 0;
          if (at < end && (MODE == kForce ? at != u : at > u)) {
            const double4 o = a.pack[at];
            double dx = home.x - o.x, dy = home.y - o.y, dz = home.z - o.z;
            dx = fma(-a.g.L[0], rint(dx * a.invL[0]), dx);
            dy = fma(-a.g.L[1], rint(dy * a.invL[1]), dy);
            dz = fma(-a.g.L[2], rint(dz * a.invL[2]), dz);
            const double t = near + o.w;
            hit = fma(dz, dz, fma(dy, dy, dx * dx)) < t * t;
            if (hit) {
              const int mo = a.sid[at];
              first = a.uniLen > 0 ? mo * a.uniLen : a.molStart[mo];
              n = a.uniLen > 0 ? a.uniLen : a.molStart[mo + 1] - first;
            }
          }
          at += 16;
          // the near molecules' atoms, in lane order
          const uint64_t mask = __ballot(hit);
          if (mask == 0) continue;
          int before, all;
          if (a.uniLen > 0) {
            before = __popcll(mask & ((uint64_t(1) << lane) - 1)) * a.uniLen;
            all = __popcll(mask) * a.uniLen;
          } else {
            int incl = n;
#pragma unroll
            for (int d = 1; d < kWave; d <<= 1) {
              const int x = __shfl_up(incl, d);
              if (lane >= d) incl += x;
            }
            before = incl - n;
            all = __builtin_amdgcn_readlane(incl, kWave - 1);
          }
          for (int t = 0; t < n; ++t) list[count + before + t] = first + t;
          count += all;
        }
        if (count == 0) break;
        // one listed atom per lane against the home atoms
        const int n = min(count, kWave);
        const bool valid = lane < n;
        count -= n;
        WaveSync();
        const int j = valid ? list[count + lane] : 0;
        WaveSync();
        double xj = 0, yj = 0, zj = 0, qj = 0, cdx = 0, cdy = 0, cdz = 0;
        int tj = 0;
        if (valid) {
          xj = a.x[j];
          yj = a.y[j];
          zj = a.z[j];
          qj = MODE == kVirial ? a.q[j] : a.q[j] * kQQFact;
          tj = a.type[j] * a.ntypes;
          if (MODE == kVirial) {
            const int mj = a.mol[j];
            cdx = MinImage(hcx - a.cx[mj], a.g.L[0], a.g.half[0]);
            cdy = MinImage(hcy - a.cy[mj], a.g.L[1], a.g.half[1]);
            cdz = MinImage(hcz - a.cz[mj], a.g.L[2], a.g.half[2]);
          }
        }
#pragma unroll 1
        for (int p = 0; p < nh; ++p) {
          const HomeAtom h = homes[w][p];
          const int ht = __builtin_amdgcn_readfirstlane(htype[w][p]);
          double dx = h.x - xj, dy = h.y - yj, dz = h.z - zj;
          dx = fma(-a.g.L[0], rint(dx * a.invL[0]), dx);
          dy = fma(-a.g.L[1], rint(dy * a.invL[1]), dy);
          dz = fma(-a.g.L[2], rint(dz * a.invL[2]), dz);
          const double d2 = fma(dz, dz, fma(dy, dy, dx * dx));
          const bool in = valid && a.g.rCutSq > d2;
          double s = 0.0;
          if (in) {
            PairType t{0.0, 0.0, 0.0, 0.0, 0.0};
            if (ht >> 30) {
              const int idx = (ht & ~(1 << 30)) + tj;
              if (inLds)
                t = PairType{tab[0][idx], tab[1][idx], tab[2][idx], tab[3][idx], tab[4][idx]};
              else
                t = PairType{a.sigSq[idx], a.epsCn[idx], a.nHalf[idx], a.epsCn6[idx], a.nOver6[idx]};
            }
            const PairTerms e = PairEval<kE, kF, MIE>(a.g, Fresh(coefs), d2, h.q * qj, t);
            if (kE) {
              lj += e.eLJ;
              real += e.eReal;
            }
            s = e.vLJ + e.vReal;
            if (MODE == kVirial) {
              const double wx = dx * cdx, wy = dy * cdy, wz = dz * cdz;
              v[0] = fma(e.vLJ, wx, v[0]);
              v[1] = fma(e.vLJ, wy, v[1]);
              v[2] = fma(e.vLJ, wz, v[2]);
              v[3] = fma(e.vReal, wx, v[3]);
              v[4] = fma(e.vReal, wy, v[4]);
              v[5] = fma(e.vReal, wz, v[5]);
            }
          }
          if (MODE == kForce) {
#pragma unroll
            for (int i = 0; i < kHomeAtoms; ++i)
              if (p == i) {  // uniform
                f[i][0] = fma(dx, s, f[i][0]);
                f[i][1] = fma(dy, s, f[i][1]);
                f[i][2] = fma(dz, s, f[i][2]);
              }
          }
        }
      }
      if (MODE == kForce) {
#pragma unroll
        for (int p = 0; p < kHomeAtoms; ++p) {
          if (p >= nh) break;
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            const double s = WaveSum(f[p][d]);
            if (S == 1) {
              double *out = d == 0 ? a.fx : (d == 1 ? a.fy : a.fz);
              if (lane == 0) out[a0 + h0 + p] = s;
            } else if (lane == 0) {
              red[w][3 * p + d] = s;
            }
          }
        }
        if (S > 1) {
          // the slices' waves of one home run the same passes
          __syncthreads();
          if (slice == 0 && lane < 3 * nh) {
            double s = red[w][lane];
            for (int i = 1; i < S; ++i) s += red[w + i][lane];
            const int d = lane % 3;
            double *out = d == 0 ? a.fx : (d == 1 ? a.fy : a.fz);
            out[a0 + h0 + lane / 3] = s;
          }
          __syncthreads();
        }
      }
    }
  }
  if (MODE == kVirial) {
#pragma unroll
    for (int i = 0; i < 6; ++i) {
      const double s = BlockSum(v[i], bred);
      if (tid == 0) a.vpart[size_t(blockIdx.x) * 6 + i] = s;
    }
  } else {
    Partial4 part{0, 0, 0, 0};
    part.lj = BlockSum(lj, bred);
    part.real = BlockSum(real, bred);
    if (MODE == kForce) {  // every pair was met twice
      part.lj *= 0.5;
      part.real *= 0.5;
    }
    FinishPartials(part, a.partials, a.counter, a.result);
  }
}

}  // namespace

// --------------------------------------------------------------- the host --
void FreeMolCells(MolCells &c) {
  for (void *p : {(void *)c.count, (void *)c.start, (void *)c.cell, (void *)c.slot, (void *)c.tmp,
                  (void *)c.sid, c.where, c.pack, (void *)c.radBits, (void *)c.vpart})
    if (p) (void)hipFree(p);
  c = MolCells{};
}

// Cells of half the reach of two molecules or more (so a molecule's partners
// lie within two cells of its own, and the corners outside the reach are
// cut finer than with cells of the whole reach), at most kMolCellsMax.
constexpr int kMolCellsMax = 1 << 15;

static void MolGrid(const gomc_box *b, int n[3], double cs[3]) {
  const double rc = std::sqrt(b->geom.rCutSq);
  double w = 0.5 * 1.0001 * (rc + 2.0 * b->molRadius);
  for (;;) {
    double cells = 1.0;
    for (int d = 0; d < 3; ++d) {
      n[d] = int(std::max(1.0, std::min(double(kMolCellsMax), std::floor(b->geom.L[d] / w))));
      cs[d] = b->geom.L[d] / n[d];
      cells *= n[d];
    }
    if (cells <= kMolCellsMax) return;
    w *= 1.25;
  }
}

// The box's molecules in cells, for the current coordinates; launched on the
// box's stream, not waited for.
static int BuildMolCells(gomc_box *b, PairArgs *out) {
  MolCells &c = b->mc;
  MolCellArgs a;
  MolGrid(b, a.n, a.cs);
  a.ncell = a.n[0] * a.n[1] * a.n[2];
  if (!c.cell) {
    const size_t n = size_t(b->nmols);
    bool ok = hipMalloc(&c.cell, sizeof(int) * n) == hipSuccess;
    ok &= hipMalloc(&c.slot, sizeof(int) * n) == hipSuccess;
    ok &= hipMalloc(&c.tmp, sizeof(int) * n) == hipSuccess;
    ok &= hipMalloc(&c.sid, sizeof(int) * n) == hipSuccess;
    ok &= hipMalloc(&c.where, sizeof(double4) * n) == hipSuccess;
    ok &= hipMalloc(&c.pack, sizeof(double4) * n) == hipSuccess;
    ok &= hipMalloc(&c.radBits, sizeof(unsigned long long) * 2) == hipSuccess;
    if (!ok) {
      FreeMolCells(c);
      return Fail(b, GOMC_ERR_HIP, "molecule cell allocation failed");
    }
    HIP_TRY(b, hipMemsetAsync(c.radBits, 0, sizeof(unsigned long long) * 2, b->stream));
  }
  if (a.ncell > c.cap) {
    for (int **p : {&c.count, &c.start}) {
      if (*p) (void)hipFree(*p);
      *p = nullptr;
    }
    c.cap = 0;
    HIP_TRY(b, hipMalloc(&c.count, sizeof(int) * a.ncell));
    HIP_TRY(b, hipMalloc(&c.start, sizeof(int) * (a.ncell + 1)));
    HIP_TRY(b, hipMemsetAsync(c.count, 0, sizeof(int) * a.ncell, b->stream));
    c.cap = a.ncell;
  }
  a.g = b->geom;
  a.x = b->x;
  a.y = b->y;
  a.z = b->z;
  a.mol = b->mol;
  a.molStart = b->molStartDev;
  a.nmols = b->nmols;
  a.count = c.count;
  a.start = c.start;
  a.cell = c.cell;
  a.slot = c.slot;
  a.tmp = c.tmp;
  a.where = static_cast<double4 *>(c.where);
  a.pack = static_cast<double4 *>(c.pack);
  a.sid = c.sid;
  a.radBits = c.radBits;
  const dim3 grid((b->nmols + kBlock - 1) / kBlock);
  hipLaunchKernelGGL(MolPlaceKernel, grid, dim3(kBlock), 0, b->stream, a);
  hipLaunchKernelGGL(MolScanKernel, dim3(1), dim3(1024), 0, b->stream, a);
  hipLaunchKernelGGL(MolScatterKernel, grid, dim3(kBlock), 0, b->stream, a);
  hipLaunchKernelGGL(MolSortKernel, grid, dim3(kBlock), 0, b->stream, a);
  HIP_TRY(b, hipGetLastError());
  PairArgs &p = *out;
  p = PairArgs{};
  p.g = b->geom;
  for (int d = 0; d < 3; ++d) {
    p.invL[d] = 1.0 / b->geom.L[d];
    p.n[d] = a.n[d];
    p.cs[d] = a.cs[d];
  }
  p.rCut = std::sqrt(b->geom.rCutSq);
  p.x = b->x;
  p.y = b->y;
  p.z = b->z;
  p.q = b->q;
  p.type = b->type;
  p.molStart = b->molStartDev;
  p.sigSq = b->tSigSq;
  p.epsCn = b->tEpsCn;
  p.nHalf = b->tNHalf;
  p.epsCn6 = b->tEpsCn6;
  p.nOver6 = b->tNOver6;
  p.ntypes = b->ntypes;
  p.nmols = b->nmols;
  p.uniLen = b->natoms == b->nmols * b->maxMolAtoms ? b->maxMolAtoms : 0;
  p.ncell = a.ncell;
  p.start = c.start;
  p.sid = c.sid;
  p.pack = a.pack;
  p.radBits = c.radBits;
  return GOMC_OK;
}

// Waves per home molecule: four while one would leave the chip's 1024 SIMDs
// with less than three waves each.
constexpr int kPairOneWave = 3072;

template <int MODE, bool MIE>
static void LaunchPairsAs(const PairArgs &a, int blocks, bool split, hipStream_t s) {
  if (split)
    hipLaunchKernelGGL((PairKernel<MODE, kPairWaves, MIE>), dim3(blocks), dim3(kPairThreads), 0, s, a);
  else
    hipLaunchKernelGGL((PairKernel<MODE, 1, MIE>), dim3(blocks), dim3(kPairThreads), 0, s, a);
}

template <int MODE>
static hipError_t LaunchPairs(const gomc_box *b, const PairArgs &a, int blocks, bool split) {
  // any other exponent than 12 brings pow's registers into the kernel
  bool mie = false;
  for (double h : b->nHalf) mie = mie || h != 6.0;
  if (mie)
    LaunchPairsAs<MODE, true>(a, blocks, split, b->stream);
  else
    LaunchPairsAs<MODE, false>(a, blocks, split, b->stream);
  return hipGetLastError();
}

static int PairBlocks(const gomc_box *b, bool *split) {
  *split = b->nmols < kPairOneWave;
  return *split ? b->nmols : (b->nmols + kPairWaves - 1) / kPairWaves;
}

int BoxInter(gomc_box *b, double *lj, double *real) {
  PairArgs a;
  int rc = BuildMolCells(b, &a);
  bool split;
  const int blocks = PairBlocks(b, &split);
  if (!rc) rc = EnsurePartials(b, blocks);
  if (rc) return rc;
  a.partials = b->partials;
  a.counter = b->counter;
  a.result = b->devRes;
  HIP_TRY(b, LaunchPairs<kEnergy>(b, a, blocks, split));
  rc = Sync(b);
  if (rc) return rc;
  *lj = b->hostRes[0];
  *real = b->hostRes[1];
  return GOMC_OK;
}

// Pair energies (hostRes[0], [1] once the stream is done) and the atoms'
// forces; not waited for.
int PairForces(gomc_box *b, double *const f[3]) {
  PairArgs a;
  int rc = BuildMolCells(b, &a);
  bool split;
  const int blocks = PairBlocks(b, &split);
  if (!rc) rc = EnsurePartials(b, blocks);
  if (rc) return rc;
  a.fx = f[0];
  a.fy = f[1];
  a.fz = f[2];
  a.partials = b->partials;
  a.counter = b->counter;
  a.result = b->devRes;
  HIP_TRY(b, LaunchPairs<kForce>(b, a, blocks, split));
  return GOMC_OK;
}

// Per-block pair virials [blocks][6] (LJ xx yy zz, real xx yy zz, the latter
// without the Coulomb constant) about the centres com; not waited for.
int PairVirials(gomc_box *b, double *const com[3], const double **vpart, int *nblocks) {
  PairArgs a;
  int rc = BuildMolCells(b, &a);
  if (rc) return rc;
  bool split;
  const int blocks = PairBlocks(b, &split);
  MolCells &c = b->mc;
  if (size_t(blocks) > c.vcap) {
    if (c.vpart) (void)hipFree(c.vpart);
    c.vpart = nullptr;
    c.vcap = 0;
    HIP_TRY(b, hipMalloc(&c.vpart, sizeof(double) * 6 * blocks));
    c.vcap = blocks;
  }
  a.cx = com[0];
  a.cy = com[1];
  a.cz = com[2];
  a.mol = b->mol;
  a.vpart = c.vpart;
  HIP_TRY(b, LaunchPairs<kVirial>(b, a, blocks, split));
  *vpart = c.vpart;
  *nblocks = blocks;
  return GOMC_OK;
}

}  // namespace gomc
