// Host check of log_wide (spectral-bslpm_amd/csrc/fasttab.hpp) against the
// long-double logarithm over its range [2^-30, 2 + 2^-5): random arguments, both
// sides of every cell boundary, near 1 and just above 2.  Fails above 0.75 ulp
// where |log x| > 1/4, above 2^-55 elsewhere (half an ulp of 1/4 is 2^-55) and above
// 2^-58 within 1e-3 of 1, and where log_wide_cell does not tell the range's outside.
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

#include "fasttab.hpp"

using namespace sbslpm;

int main() {
  std::vector<LogTabEntry> tab(kLogWideSize);
  build_log_wide_table(tab.data());
  double ulps = 0, small = 0, one = 0;
  auto check = [&](double x) {
    const uint32_t h = log_wide_cell(x);
    if (h >= kLogWideSpan) return;
    const long double ref = logl((long double)x);
    const double a = std::fabs((double)ref), err = (double)fabsl(log_wide(x, h, tab.data(), 1.0 / 7.0) - ref);
    if (a > 0.25)
      ulps = std::max(ulps, err / (std::nextafter(a, INFINITY) - a));
    else
      small = std::max(small, err);
    if (std::fabs(x - 1.0) < 1e-3) one = std::max(one, err);
  };
  std::mt19937_64 g(1);
  std::uniform_real_distribution<double> e(-30.0, 1.0), lin(0.0, 2.0);
  for (int i = 0; i < 2000000; ++i) {
    check(std::exp2(e(g)));
    check(lin(g));
  }
  for (int i = 0; i < kLogWideSize; ++i) {
    const double lo = std::ldexp(1.0 + (i % 64) / 64.0, i / 64 - 30);
    for (double x : {lo, std::nextafter(lo, 0.0), std::nextafter(lo, 4.0)}) check(x);
  }
  for (int i = -1000; i <= 1000; ++i) check(1.0 + i * 1e-9);
  std::uniform_real_distribution<double> near(-1e-3, 1e-3);
  for (int i = 0; i < 1000000; ++i) check(1.0 + near(g));
  bool range = true;
  for (double x : {0.0, -0.0, -1e-16, -1.0, 1e-300, std::nextafter(0x1p-30, 0.0), 2.04, 1e300, (double)INFINITY,
                   -(double)INFINITY, (double)NAN})
    range = range && log_wide_cell(x) >= kLogWideSpan;
  for (double x : {0x1p-30, 1.0, 2.0, std::nextafter(2.0, 3.0), 2.03}) range = range && log_wide_cell(x) < kLogWideSpan;
  std::printf("log_wide: %.3f ulp where |log| > 1/4, %.3g elsewhere, %.3g (2^%.2f) near 1, range %d\n", ulps, small, one,
              std::log2(one), (int)range);
  return ulps <= 0.75 && small <= 0x1p-55 && one <= 0x1p-58 && range ? 0 : 1;
}
