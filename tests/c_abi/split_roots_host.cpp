// Host check of SplitRoots (no GPU): every root against the one evaluated by
// itself. Each is rounded once from long double, so they differ by at most one
// unit in the last place of [0.5, 1). Prints the roots compared.
#include <algorithm>
#include <cmath>
#include <cstdio>

#include "../../perf-libs-fft_amd/csrc/plan.hpp"

int main() {
  long count = 0;
  for (int64_t n : {1, 2, 3, 7, 12, 64, 96, 100, 1000, 4096, 12288, 65536, 98304, 131072, 1048576}) {
    const plf::SplitRoots root(n);
    double worst = 0;
    for (int64_t e = 0; e < n; ++e) {
      double re, im, z[2];
      plf::unit_root(e, n, &re, &im);
      root(e, z);
      worst = std::max(worst, std::max(std::fabs(z[0] - re), std::fabs(z[1] + im)));
      ++count;
    }
    if (!(worst <= std::ldexp(1.0, -53))) {
      std::printf("order %lld: %g\n", (long long)n, worst);
      return 1;
    }
  }
  std::printf("%ld\n", count);
  return 0;
}
