// Prints the relative error of the batched kernel's Coulomb table against
// extended-precision values: worst and root mean square over a dense set of
// r^2 up to the cutoff, row edges included, and the smallest r^2 tabulated.
#include <algorithm>
#include <cstdio>
#include <cstdlib>

#include "../gomc_amd/csrc/coul_table.hpp"

using namespace gomc;

int main(int argc, char **argv) {
  const double tol = atof(argv[1]), rcut = atof(argv[2]);
  const bool ewald = atoi(argv[3]) != 0;
  const double alpha = std::sqrt(-std::log(tol)) / rcut, rc2 = rcut * rcut;
  CoulTable tab;
  MakeCoulTable(alpha, ewald, rc2, &tab);
  std::vector<TabPair> pairs(kTabWords / 2 + 1);
  std::memcpy(pairs.data(), tab.c.data(), sizeof(double) * kTabWords);
  const double *tail = reinterpret_cast<const double *>(pairs.data());
  double worst = 0.0, sum = 0.0, t, first = 0.0;
  long count = 0;
  auto test = [&](double d2) {
    if (d2 >= rc2) return;
    const int row = TabRow(d2, tab.base, &t);
    if (row < 0 || row >= kTabRows) {
      std::printf("not tabulated: %.17g\n", d2);
      std::exit(1);
    }
    const double f = TabValue(pairs.data(), tail, row, t);
    const long double r = sqrtl((long double)d2);
    const long double e = ewald ? erfcl((long double)alpha * r) / r : 1.0L / r;
    const double err = std::fabs(double((f - e) / e));
    worst = std::max(worst, err);
    sum += err * err;
    ++count;
  };
  for (int row = 0; row < kTabRows; ++row) {
    const uint64_t lo = uint64_t(tab.base + row) << (kTabShift + 32),
                   hi = uint64_t(tab.base + row + 1) << (kTabShift + 32);
    double from, to;
    std::memcpy(&from, &lo, 8);
    std::memcpy(&to, &hi, 8);
    if (row == 0) first = from;
    test(from);
    test(std::nextafter(to, from));
    for (int s = 1; s < 40; ++s) test(from + (to - from) * (s + 0.37 * ((row * 7 + s) % 5) / 5.0) / 41.0);
  }
  test(std::nextafter(rc2, 0.0));
  std::printf("%.3e %.3e %.17g %ld\n", worst, std::sqrt(sum / count), first, count);
  return 0;
}
