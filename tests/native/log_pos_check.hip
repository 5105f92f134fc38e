// Host-side check of log_pos and div_normal (botorch_amd/csrc/bta_common.h) against
// the C library in long double: log over the whole positive range and densely
// around 1, the quotient over the Pareto denominators.  Prints the largest errors
// in units of the last place; exits 1 if one exceeds 1.
#include <cmath>
#include <cstdio>
#include <limits>
#include <random>

#include "../../botorch_amd/csrc/bta_common.h"

static double ulps(double got, long double ref) {
  const double r = std::fabs((double)ref);
  const double u = std::nextafter(r, std::numeric_limits<double>::infinity()) - r;
  return (double)(std::fabs((long double)got - ref) / u);
}

int main() {
  double worst = 0.0, worst_div = 0.0;
  std::mt19937_64 g(1);
  std::uniform_real_distribution<double> U(0.0, 1.0);
  auto check = [&](double x) {
    const double e = ulps(bta::log_pos(x), std::log((long double)x));
    if (e > worst) worst = e;
  };
  for (int i = 0; i < 3000000; ++i) {
    check(std::exp2(2046.0 * U(g) - 1022.0));  // every binade
    check(0.5 + 2.0 * U(g));                   // around 1, both branches of f
    check(1.0 + 32.0 * U(g));                  // the Pareto sums
    check(1.0 + std::exp2(-52.0 * U(g)));      // just above 1
    check(1.0 - std::exp2(-1.0 - 51.0 * U(g)));
    const double n = U(g) * 4.0 - 2.0, d = 1.0 + std::exp2(300.0 * U(g));
    const double e = ulps(bta::div_normal(n, d), (long double)n / (long double)d);
    if (e > worst_div) worst_div = e;
  }
  const double inf = std::numeric_limits<double>::infinity();
  const bool special = bta::log_pos(1.0) == 0.0 && bta::log_pos(inf) == inf &&
                       std::isnan(bta::log_pos(std::numeric_limits<double>::quiet_NaN())) &&
                       std::fabs(bta::log_pos(5e-324) - std::log(5e-324)) < 1e-12;
  std::printf("log %.3f ulp, div %.3f ulp, special %d\n", worst, worst_div, (int)special);
  return (worst <= 1.0 && worst_div <= 1.0 && special) ? 0 : 1;
}
