// Device helpers shared by the gfx950 kernels: minimum image, the Mie/LJ
// and erfc-Coulomb pair terms, Philox4x64-10, and wave64/workgroup
// reductions in a fixed order (so a sum does not depend on timing).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "erfcx_poly.hpp"

namespace gomc {

constexpr double kQQFact = 167103.208067979;  // lib/NumLib.h:22
constexpr int kWave = 64;

// BoxDimensions::MinImageSigned (src/BoxDimensions.h:169-175): the same
// single add or subtract, chosen by selects rather than branches.
__device__ __forceinline__ double MinImage(double d, double ax, double half) {
  const double down = d - ax, up = d + ax;
  return d > half ? down : (d < -half ? up : d);
}

// BoxDimensions::WrapPBC (src/BoxDimensions.cpp:261-296).
__host__ __device__ __forceinline__ double Wrap(double v, double ax) {
  if (v >= ax)
    v -= ax;
  else if (v < 0)
    v += ax;
  return v;
}

// BoxDimensions::UnwrapPBC (src/BoxDimensions.cpp:298-320).
__host__ __device__ __forceinline__ double Unwrap(double v, double ref, double ax,
                                                  double half) {
  if (fabs(ref - v) > half) {
    if (ref < half)
      v -= ax;
    else
      v += ax;
  }
  return v;
}

// Orthogonal box geometry and cutoffs passed by value to every kernel.
struct BoxGeom {
  double L[3], half[3];
  double rCutSq;      // box cutoff max(Rcut, RcutCoulomb) squared
  double rCutLJSq;    // Rcut squared (FFParticle::CalcEn gate)
  double rCutCoulSq;  // RcutCoulomb squared (FFParticle::CalcCoulomb gate)
  double rCutLowSq;   // RcutLow squared (overlap test)
  double alpha;       // Ewald alpha
  int ewald, elect;
};

// Squared minimum-image distance in the reference's operation order
// (InRcut, src/BoxDimensions.h:231-261): each component min-imaged, then
// x*x + y*y + z*z left to right.  Files are built without FMA contraction.
__device__ __forceinline__ double DistSq(const BoxGeom &g, double ax, double ay, double az,
                                         double bx, double by, double bz) {
  double dx = MinImage(ax - bx, g.L[0], g.half[0]);
  double dy = MinImage(ay - by, g.L[1], g.half[1]);
  double dz = MinImage(az - bz, g.L[2], g.half[2]);
  return dx * dx + dy * dy + dz * dz;
}

// Mixed precision (FP32 pair terms and phases, FP64 accumulation): the
// same terms in FP32 from the FP64 squared distance.
__device__ __forceinline__ double CoulombEnergyF32(const BoxGeom &g, double distSq, double qiqj) {
  const float d = sqrtf(float(distSq));
  if (g.ewald) return double(float(qiqj) * erfcf(float(g.alpha) * d) / d);
  return double(float(qiqj) / d);
}

__device__ __forceinline__ double LJEnergyF32(double distSq, double sigmaSq, double epsCn,
                                              double nHalf) {
  const float rRat2 = float(sigmaSq) / float(distSq);
  const float att = rRat2 * rRat2 * rRat2;
  const float rep = (nHalf == 6.0) ? att * att : powf(rRat2, float(nHalf));
  return double(float(epsCn) * (rep - att));
}

// sincos(ang) in FP32 after reducing the FP64 argument to [-pi, pi).
__device__ __forceinline__ void SincosF32(double ang, double *s, double *c) {
  const double turns = ang * (0.5 * M_1_PI);
  const float red = float((turns - rint(turns)) * (2.0 * M_PI));
  float sf, cf;
  sincosf(red, &sf, &cf);
  *s = sf;
  *c = cf;
}

// ---------------------------------------------------------- Philox -------
// Philox4x64-10 (Salmon et al. 2011; the generator the reference vendors as
// lib/Random123/philox.h): 10 rounds of two 64x64->128 multiplies with the
// published multipliers, key bumped by the Weyl constants between rounds.
struct U64x4 {
  uint64_t v[4];
};

__host__ __device__ __forceinline__ void MulHiLo(uint64_t a, uint64_t b, uint64_t &hi,
                                                 uint64_t &lo) {
#if defined(__HIP_DEVICE_COMPILE__)
  lo = a * b;
  hi = __umul64hi(a, b);
#else
  unsigned __int128 p = (unsigned __int128)a * b;
  hi = uint64_t(p >> 64);
  lo = uint64_t(p);
#endif
}

__host__ __device__ __forceinline__ U64x4 Philox(uint64_t c0, uint64_t c1, uint64_t c2,
                                                 uint64_t c3, uint64_t k0, uint64_t k1) {
  const uint64_t M0 = 0xD2E7470EE14C6C93ull, M1 = 0xCA5A826395121157ull;
  const uint64_t W0 = 0x9E3779B97F4A7C15ull, W1 = 0xBB67AE8584CAA73Bull;
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    if (r) {
      k0 += W0;
      k1 += W1;
    }
    uint64_t hi0, lo0, hi1, lo1;
    MulHiLo(M0, c0, hi0, lo0);
    MulHiLo(M1, c2, hi1, lo1);
    uint64_t n0 = hi1 ^ c1 ^ k0, n2 = hi0 ^ c3 ^ k1;
    c0 = n0;
    c1 = lo1;
    c2 = n2;
    c3 = lo0;
  }
  U64x4 o;
  o.v[0] = c0;
  o.v[1] = c1;
  o.v[2] = c2;
  o.v[3] = c3;
  return o;
}

// r123::u01<double> for a 64-bit word (lib/Random123/uniform.hpp:174-183):
// x * 2^-64 + 2^-65, the product exact, one rounding in the add.
__host__ __device__ __forceinline__ double U01(uint64_t v) {
  return double(v) * 0x1p-64 + 0x1p-65;
}

// erfcx(x) = exp(x^2) erfc(x) for x >= 4 from Laplace's continued fraction
// erfc(x) = exp(-x^2) / sqrt(pi) / (x + (1/2) / (x + 1 / (x + (3/2) / ...))),
// evaluated from the tail, 24 levels: relative error about 4e-16 for every
// x >= 4.  Two live values, where libm's erfc holds dozens of registers.
__device__ __forceinline__ double ErfcxTail(double x) {
  double f = x;
#pragma unroll 1
  for (int n = 24; n >= 1; --n) f = x + (0.5 * n) / f;
  return 1.0 / (1.7724538509055160273 * f);
}

// x^h for the Mie repulsion (sigma^2/r^2)^(n/2): whole and half-integer h
// up to 32 by repeated squaring (and one sqrt), within a few ulps of pow;
// any other h as exp(h log x).
__device__ __forceinline__ double MiePow(double x, double h) {
  const double twice = 2.0 * h;
  if (h > 0.0 && h <= 32.0 && twice == floor(twice)) {
    int k = int(h);
    double r = 1.0, b = x;
    while (k) {
      if (k & 1) r *= b;
      b *= b;
      k >>= 1;
    }
    return twice == 2.0 * floor(h) ? r : r * sqrt(x);
  }
  return exp(h * log(x));
}

// 1/sqrt(d2) to double precision: the hardware estimate and two Newton
// steps y <- y (3/2 - d2 y^2 / 2).
__device__ __forceinline__ double Rsqrt64(double d2) {
  const double h = 0.5 * d2;
  double y = __builtin_amdgcn_rsq(d2);
  y = y * fma(-h * y, y, 1.5);
  y = y * fma(-h * y, y, 1.5);
  return y;
}

// Coefficients of the pair terms, highest power first: the Taylor series of
// e^r to r^13 / 13!, then erfcx's fitted polynomial.  Read through the scalar
// cache into scalar registers each time they are used (Coefs): they cost the
// vector units nothing there, where LDS would feed four SIMDs one broadcast at
// a time and 43 held values would not leave room for four waves a SIMD.
constexpr int kExpDeg = 13;
struct CoefTable {
  double c[kExpDeg + 1 + kErfcxDeg + 1];
};
constexpr CoefTable MakeCoefs() {
  CoefTable t{};
  double f = 1.0;
  for (int k = 0; k <= kExpDeg; ++k) {
    if (k > 0) f *= k;
    t.c[kExpDeg - k] = 1.0 / f;
  }
  for (int k = 0; k <= kErfcxDeg; ++k) t.c[kExpDeg + 1 + k] = kErfcxPoly[kErfcxDeg - k];
  return t;
}
static __constant__ CoefTable coefTable = MakeCoefs();
typedef const double __attribute__((address_space(4))) *Coefs;
__device__ __forceinline__ Coefs GetCoefs() { return (Coefs)coefTable.c; }
// The same pointer, as far as the compiler knows another one: what is read
// through it is not kept from one use to the next.
__device__ __forceinline__ Coefs Fresh(Coefs c) {
  asm volatile("" : "+s"(c));
  return c;
}

// a b + c with c from scalar registers.  Written out because the compiler
// otherwise takes the two-operand form and first moves every coefficient to
// vector registers, two more instructions for each multiply-add.
__device__ __forceinline__ double FmaS(double a, double b, double c) {
  double d;
  asm("v_fma_f64 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "s"(c));
  return d;
}

// e^y for y in [-700, 0]: y = n ln 2 + r with |r| <= ln 2 / 2, the Taylor
// series of e^r (truncation 4e-18), scaled by 2^n.
__device__ __forceinline__ double ExpNeg(Coefs c, double y) {
  const double n = rint(y * M_LOG2E);
  double r = fma(-n, 0x1.62e42fefa39efp-1, y);  // ln 2 to 53 bits, and the rest
  r = fma(-n, 0x1.abc9e3b39803fp-56, r);
  double p = c[0];
#pragma unroll
  for (int k = 1; k <= kExpDeg; ++k) p = FmaS(p, r, c[k]);
  return ldexp(p, int(n));
}

// sigma^2 / d2 to the last place from ir = 1 / sqrt(d2): powers of it multiply
// its error, so one correction is spent on it rather than on 1 / d2.
__device__ __forceinline__ double LJRatio(double sigmaSq, double d2, double ir) {
  const double ir2 = ir * ir, x = sigmaSq * ir2;
  return fma(fma(-d2, x, sigmaSq), ir2, x);
}

// The Mie repulsion for exponents other than 12, out of line where its
// registers would weigh on a pair loop.
static __device__ __noinline__ double PowOutOfLine(double x, double h) { return pow(x, h); }

// Pair terms at precision P (FFParticle::CalcEn / CalcCoulomb,
// src/FFParticle.cpp:295-399).  FP64: one reciprocal square root (a
// Newton-refined estimate, then one correction each for r and sigma^2 / r^2, to
// the last place) stands for the root and the divisions, e^-x^2 and erfcx are
// polynomials whose coefficients are scalar operands, and for the exponent 12
// nothing is called: a call would save and restore the registers of the pair
// loops.  LIBM: libm's erfc, whose error is a tenth of the polynomial's 3e-15.
template <int P, bool LIBM = false>
__device__ __forceinline__ void PairTermsDev(const BoxGeom &g, Coefs cf, double d2, double qiqj,
                                             double sigmaSq, double epsCn, double nHalf,
                                             double sign, double &lj, double &real) {
  const bool coul = g.elect && qiqj != 0.0 && !(g.rCutCoulSq < d2);
  const bool inLJ = !(g.rCutLJSq < d2);
  if (P) {
    if (coul) real += sign * CoulombEnergyF32(g, d2, qiqj);
    if (inLJ) lj += sign * LJEnergyF32(d2, sigmaSq, epsCn, nHalf);
    return;
  }
  d2 = fmax(d2, 0x1p-1022);  // coincident atoms: huge, not 0 x inf
  const double ir = Rsqrt64(d2);
  if (coul) {
    double e = qiqj * ir;
    if (LIBM && g.ewald) {
      double dist = d2 * ir;
      dist = fma(fma(-dist, dist, d2), 0.5 * ir, dist);
      e *= erfc(g.alpha * dist);
    } else if (g.ewald) {
      double dist = d2 * ir;
      dist = fma(fma(-dist, dist, d2), 0.5 * ir, dist);
      const double x = g.alpha * dist;
      double ex;
      if (x <= kErfcxUse) {
        const double u = (x - kErfcxMid) * kErfcxInvHalf;
        ex = cf[kExpDeg + 1];
#pragma unroll
        for (int k = 1; k <= kErfcxDeg; ++k) ex = FmaS(ex, u, cf[kExpDeg + 1 + k]);
      } else {
        ex = ErfcxTail(x);
      }
      e *= ExpNeg(cf, fmax(-(x * x), -700.0)) * ex;
    }
    real += sign * e;
  }
  if (inLJ) {
    const double rRat2 = LJRatio(sigmaSq, d2, ir);
    const double att = rRat2 * rRat2 * rRat2;
    double rep = att * att;
    if (nHalf != 6.0) rep = LIBM ? pow(rRat2, nHalf) : PowOutOfLine(rRat2, nHalf);
    lj += sign * (epsCn * (rep - att));
  }
}

// Sum over the wave in a fixed tree, valid in lane 63: four steps within rows
// of 16 lanes, then the rows.  Lane moves are VALU operations here, a shuffle
// through LDS is several times their latency.
__device__ __forceinline__ double WaveSumDpp(double v) {
  auto step = [](double x, auto ctrl, auto rows) {
    const uint64_t u = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = __builtin_amdgcn_update_dpp(0u, uint32_t(u), decltype(ctrl)::value,
                                                    decltype(rows)::value, 0xf, false);
    const uint32_t hi = __builtin_amdgcn_update_dpp(0u, uint32_t(u >> 32), decltype(ctrl)::value,
                                                    decltype(rows)::value, 0xf, false);
    return x + __builtin_bit_cast(double, (uint64_t(hi) << 32) | lo);
  };
  v = step(v, std::integral_constant<int, 0x111>{}, std::integral_constant<int, 0xf>{});  // row_shr:1
  v = step(v, std::integral_constant<int, 0x112>{}, std::integral_constant<int, 0xf>{});
  v = step(v, std::integral_constant<int, 0x114>{}, std::integral_constant<int, 0xf>{});
  v = step(v, std::integral_constant<int, 0x118>{}, std::integral_constant<int, 0xf>{});
  v = step(v, std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{});  // row_bcast:15
  v = step(v, std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{});  // row_bcast:31
  return v;
}

// The pair terms and phases at precision P: 0 is FP64 throughout, 1 the
// FP32 forms above (sums stay FP64 in every caller).
template <int P>
__device__ __forceinline__ void Sincos(double ang, double *s, double *c) {
  if (P)
    SincosF32(ang, s, c);
  else
    sincos(ang, s, c);
}

// ------------------------------------------------------- reductions -------
template <typename T>
__device__ __forceinline__ T WaveSum(T v) {
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) v += __shfl_down(v, off, kWave);
  return v;  // valid in lane 0
}

// Sum over the workgroup; the result is valid in thread 0.  `lds` holds one
// slot per wave.  Order: lanes by tree within a wave, then waves in index
// order.  Contains __syncthreads().
template <typename T>
__device__ __forceinline__ T BlockSum(T v, T *lds) {
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int nwaves = (blockDim.x + kWave - 1) / kWave;
  v = WaveSum(v);
  if (lane == 0) lds[wave] = v;
  __syncthreads();
  T r = T(0);
  if (threadIdx.x == 0)
    for (int w = 0; w < nwaves; ++w) r += lds[w];
  __syncthreads();
  return r;
}

// Four sums over the workgroup with one barrier, valid in every lane of the
// first wave: each wave's by lane moves, then one value a lane.
__device__ __forceinline__ void BlockSum4(double (&v)[4], double (*lds)[4]) {
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int nwaves = blockDim.x / kWave;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = WaveSumDpp(v[i]);
  if (lane == kWave - 1)
#pragma unroll
    for (int i = 0; i < 4; ++i) lds[wave][i] = v[i];
  __syncthreads();
  if (wave == 0) {
    double r = (lane >> 2) < nwaves ? lds[lane >> 2][lane & 3] : 0.0;
#pragma unroll
    for (int off = kWave / 2; off >= 4; off >>= 1) r += __shfl_down(r, off, kWave);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = __shfl(r, i, kWave);
  }
}

}  // namespace gomc
