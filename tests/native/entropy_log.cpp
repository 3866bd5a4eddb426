// entropy_log.cpp -- the entropic solve's logarithms against the 80-bit library logarithm
// (built and run by tests/test_entropy_log.py).
//
// Bound: the quotient s is good to 1.5 units in the last place, the polynomial's fused
// sum and the addition of k ln 2 add one each, so 4 units of the result cover both.
#include <cfloat>
#include <cmath>
#include <cstdio>

#include "entropy_log.hpp"

int main() {
  int values = 0, failures = 0;
  double worst[2] = {0.0, 0.0};
  auto check = [&](int which, double x, double got, long double want) {
    ++values;
    const double unit = DBL_EPSILON * (double)fabsl(want) + DBL_MIN;
    const double units = (double)fabsl((long double)got - want) / unit;
    if (units > worst[which]) worst[which] = units;
    if (!(units <= 4.0) && ++failures <= 10)
      std::printf("FAIL %s(%.17g) = %.17g, off by %g units\n", which ? "log1p_positive" : "log_or_nan",
                  x, got, units);
  };
  // from the smallest normal number to beyond any f / w, denser around 1
  for (double e = -1022.0; e <= 20.0; e += 0.00731) {
    const double v = std::exp2(e);
    check(0, v, lbm::log_or_nan(v), logl((long double)v));
  }
  for (double v : {4.9406564584124654e-324, 1e-320, 1e-310, 1e-300, 1e-20, 1e-17, 0x1p-53, 0.5,
                   0.70710678118654746, 0.70710678118654757, 0.9999999999999999, 1.0,
                   1.0000000000000002, 1.4142135623730949, 1.4142135623730951})
    check(0, v, lbm::log_or_nan(v), logl((long double)v));
  for (int j = -20000; j <= 20000; ++j) {
    const double y = j / 20001.0, small = y * 1e-9;
    check(0, 1.0 + y, lbm::log_or_nan(1.0 + y), logl((long double)(1.0 + y)));
    check(1, y, lbm::log1p_positive(y), log1pl((long double)y));
    check(1, small, lbm::log1p_positive(small), log1pl((long double)small));
  }
  for (double v : {0.0, -0.0, -1e-300, -1.0})
    if (!std::isnan(lbm::log_or_nan(v))) ++failures;
  std::printf("%d values, worst %g and %g units, %d failures\n", values, worst[0], worst[1], failures);
  return failures != 0 || values < 200000;
}
