// Host-side check of div_by and log_pos (botorch_amd/csrc/bta_common.h) at the ends of
// their ranges: log_pos of the smallest and largest normal numbers, div_by for infinite,
// zero and NaN operands against the division, and its equality with the division over
// ordinary operands.  Argument: div or log.  Prints the first mismatch; exits 1 if there
// is one.
#include <cfloat>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <limits>
#include <random>

#include "../../botorch_amd/csrc/bta_common.h"

static bool same(double a, double b) {
  return (std::isnan(a) && std::isnan(b)) || (a == b && std::signbit(a) == std::signbit(b));
}

static int check_div() {
  const double inf = std::numeric_limits<double>::infinity();
  const double nan = std::numeric_limits<double>::quiet_NaN();
  int bad = 0;
  auto quot = [&](double x, double l) {
    const double got = bta::div_by(x, l, 1.0 / l), want = x / l;
    if (!same(got, want) && !bad++) std::printf("%a / %a: %a, not %a\n", x, l, got, want);
  };
  for (double l : {1.0, -3.0, 1e-100, 1e100, inf, -inf, nan})
    for (double x : {0.0, -0.0, 1.0, -7.0, 1e-150, 1e150, inf, -inf, nan}) quot(x, l);
  for (double x : {1.0, -1.0, inf, nan}) quot(x, 0.0);
  std::mt19937_64 g(3);
  std::uniform_real_distribution<double> U(-1.0, 1.0);
  for (int i = 0; i < 2000000; ++i)
    quot(std::ldexp(1.0 + std::fabs(U(g)), (int)(400 * U(g))) * (U(g) < 0 ? -1 : 1),
         std::ldexp(1.0 + std::fabs(U(g)), (int)(400 * U(g))));
  return bad;
}

static int check_log() {
  int bad = 0;
  for (double x : {DBL_MIN, DBL_MAX, std::nextafter(DBL_MAX, 0.0), 5e-324}) {
    const double got = bta::log_pos(x), want = std::log(x);
    if (!(std::fabs(got - want) <= 1.2e-13) && !bad++)  // an ulp of 709
      std::printf("log %a: %a, not %a\n", x, got, want);
  }
  return bad;
}

int main(int argc, char** argv) {
  return (argc > 1 && !std::strcmp(argv[1], "log") ? check_log() : check_div()) != 0;
}
