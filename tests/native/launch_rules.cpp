// launch_rules.cpp -- how the 2D kernel's steps are split over launches, for calls from one
// step to the largest number that lbm_step takes (built and run by
// tests/test_launch_rules.py).
#include <climits>
#include <cstdio>
#include <vector>

#include "config_rules.hpp"

int main() {
  std::vector<int> calls;
  for (int n = 1; n <= 400; ++n) calls.push_back(n);
  for (int k = 0; k < 12; ++k) calls.push_back(INT_MAX - k);
  int failures = 0;
  for (int per = 2; per <= 5; ++per)
    for (int n : calls) {
      const int launches = lbm::launches_of(n, per);
      // Every launch takes 1 to `per` steps, the last one those that are left.  A long call
      // is followed for its first launches; the rule keeps steps / launches after that.
      int left = n, to_go = launches;
      bool ok = launches >= 1 && (n - launches) % 2 == 0;
      for (int k = 0; ok && to_go > 0 && k < 1000; ++k, --to_go) {
        const int take = lbm::steps_of_next(left, to_go);
        ok = take >= 1 && take <= per && take <= left;
        left -= take;
      }
      if (to_go == 0) ok = ok && left == 0;
      else ok = ok && left >= to_go && (left - 1LL + per) / per <= to_go;
      // no more launches than the parity asks for
      ok = ok && launches - 2 < (n - 1LL + per) / per;
      if (!ok) {
        std::printf("FAIL %d steps, %d a launch: %d launches, %d left\n", n, per, launches, left);
        ++failures;
      }
    }
  std::printf("%d failures\n", failures);
  return failures != 0;
}
