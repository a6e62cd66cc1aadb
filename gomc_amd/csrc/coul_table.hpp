// The Coulomb factor erfc(alpha r) / r (1 / r without Ewald) of the batched
// kernel as a function of r^2: a polynomial of degree 8 in each 64th of an
// octave of r^2, over the eight octaves that end at the first power of two not
// below the Coulomb cutoff squared.  Row and offset come from the bits of r^2,
// and eight multiply-adds stand for the reciprocal square root, the exponential
// and the 28th-degree erfcx (75 instructions).  Below the first octave (r under
// a sixteenth to an eleventh of the cutoff) the factor is computed directly.
//
// Made on the host, once per alpha and cutoff, from the values at the rows'
// nine Chebyshev nodes in extended precision, so that the coefficients carry
// their own rounding and nothing else.  Relative error against 64-bit-mantissa
// values, worst / root mean square over cutoffs of 8 to 16 A: 1.2e-15 / 1.7e-16
// at tolerance 1e-5 and 1e-6, 2.7e-15 / 2.3e-16 at 1e-10 (the polynomial form
// exp(-x^2) erfcx(x): 7.9e-15 / 1.2e-15 and 1.2e-14 / 1.8e-15).  Degree 7 leaves
// 4.5e-15 at 1e-6 and 1.4e-13 at 1e-10 where the cutoff lies just above a power
// of two, for its interpolation error.
#pragma once

#include <cmath>
#include <cstdint>
#include <cstring>
#include <vector>

#if defined(__HIPCC__)
#define COUL_HD __host__ __device__ __forceinline__
#else
#define COUL_HD inline
#endif

namespace gomc {

constexpr int kTabBits = 6, kTabOctaves = 8, kTabRows = kTabOctaves << kTabBits, kTabDeg = 8;
constexpr int kTabShift = 20 - kTabBits;           // of the high word of r^2
constexpr int kTabWords = kTabRows * (kTabDeg + 1);  // doubles of a table

// Where coefficient k of a row lies.  0..7: pairs of coefficients (16 bytes)
// change places from row to row, so that one pair of many rows is spread over
// all LDS banks (eight coefficients are a quarter of them); 8: behind all rows.
COUL_HD int TabAt(int row, int k) {
  return k < 8 ? row * 8 + (k ^ ((row >> 1) & 6)) : kTabRows * 8 + row;
}

// Row of r^2 in a table of this base (outside [0, kTabRows): not tabulated), and
// r^2 less the row's middle.
COUL_HD int TabRow(double d2, int base, double *t) {
  const uint64_t u = __builtin_bit_cast(uint64_t, d2);
  const uint32_t hi = uint32_t(u >> 32);
  const uint32_t mid = (hi & ~((1u << kTabShift) - 1)) | (1u << (kTabShift - 1));
  *t = d2 - __builtin_bit_cast(double, uint64_t(mid) << 32);
  return int(hi >> kTabShift) - base;
}

typedef double TabPair __attribute__((vector_size(16)));

// The polynomial of a row at t; `pairs` and `tail` point to the table's start.
template <typename PairPtr, typename Ptr>
COUL_HD double TabValue(PairPtr pairs, Ptr tail, int row, double t) {
  const int x = (row >> 2) & 3;
  const PairPtr c = pairs + row * 4;
  const TabPair c6 = c[3 ^ x], c4 = c[2 ^ x], c2 = c[1 ^ x], c0 = c[x];
  double f = tail[kTabRows * 8 + row];
  f = __builtin_fma(f, t, c6[1]);
  f = __builtin_fma(f, t, c6[0]);
  f = __builtin_fma(f, t, c4[1]);
  f = __builtin_fma(f, t, c4[0]);
  f = __builtin_fma(f, t, c2[1]);
  f = __builtin_fma(f, t, c2[0]);
  f = __builtin_fma(f, t, c0[1]);
  return __builtin_fma(f, t, c0[0]);
}

// ------------------------------------------------------------- the host --
struct CoulTable {
  double alpha = -1.0;
  bool ewald = false;
  int base = 0;
  std::vector<double> c;  // [kTabWords]
};

// Base of the table whose last octave ends at or beyond rCutSq.
inline int TabBase(double rCutSq) {
  int e = 0;
  const double m = std::frexp(rCutSq, &e);  // rCutSq = m 2^e, m in [1/2, 1)
  if (m == 0.5) --e;
  return (1023 + e - kTabOctaves) << kTabBits;
}

// The coefficients of the polynomial through the values at the Chebyshev nodes
// of each row (the Lagrange polynomials, expanded).
inline void MakeCoulTable(double alpha, bool ewald, double rCutSq, CoulTable *out) {
  constexpr int n = kTabDeg + 1;
  const long double pi = 3.141592653589793238462643383279502884L;
  long double node[n], m[n][n];
  for (int j = 0; j < n; ++j) node[j] = cosl((2 * j + 1) * pi / (2 * n));
  for (int j = 0; j < n; ++j) {
    long double p[n] = {1.0L}, den = 1.0L;
    int deg = 0;
    for (int i = 0; i < n; ++i) {
      if (i == j) continue;
      den *= node[j] - node[i];
      ++deg;
      for (int k = deg; k >= 0; --k)
        p[k] = (k > 0 ? p[k - 1] : 0.0L) - node[i] * (k < deg ? p[k] : 0.0L);
    }
    for (int k = 0; k < n; ++k) m[k][j] = p[k] / den;
  }
  out->alpha = alpha;
  out->ewald = ewald;
  out->base = TabBase(rCutSq);
  out->c.assign(kTabWords, 0.0);
  for (int row = 0; row < kTabRows; ++row) {
    const uint64_t place = uint64_t(out->base + row) << kTabShift;
    const uint64_t lo = place << 32, hi = (place + (1u << kTabShift)) << 32;
    double from, to;
    std::memcpy(&from, &lo, 8);
    std::memcpy(&to, &hi, 8);
    const long double half = 0.5L * ((long double)to - from), mid = from + half;
    long double v[n];
    for (int j = 0; j < n; ++j) {
      const long double r = sqrtl(mid + half * node[j]);
      v[j] = ewald ? erfcl(alpha * r) / r : 1.0L / r;
    }
    long double scale = 1.0L;
    for (int k = 0; k < n; ++k, scale /= half) {
      long double s = 0.0L;
      for (int j = 0; j < n; ++j) s += m[k][j] * v[j];
      out->c[TabAt(row, k)] = double(s * scale);
    }
  }
}

}  // namespace gomc
