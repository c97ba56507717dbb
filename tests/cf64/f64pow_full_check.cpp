// Host build of csrc/k_f64math.h: f64_pow_full against 113-bit arithmetic.
// Prints the largest error in ulp of the result over samples of each range, then
// the quotients of f64_div_by that differ from the IEEE division's.
#include <quadmath.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <initializer_list>

#include "k_f64math.h"

static double ulp_error(double v, __float128 ref) {
  int e;
  frexp((double)ref, &e);
  return fabs((double)((v - ref) / (__float128)ldexp(1.0, e - 53)));
}

int main() {
  const double rcp = 1.0 - 1.0 / (double)1.4f;  // R / cp of the energy sum
  const struct {
    double lo, hi, c;
  } range[] = {{0.01, 1.05, rcp}, {0.99, 1.01, rcp}, {1e-45, 1e38, rcp}, {0.3, 3.0, 1.4}, {0.7, 1.5, -5.3}};
  uint64_t x = 88172645463325252ull;  // xorshift
  for (auto &r : range) {
    double worst = 0.0;
    const int n = 200000;
    for (int q = 0; q < n; q++) {
      x ^= x << 13;
      x ^= x >> 7;
      x ^= x << 17;
      const double t = r.lo * pow(r.hi / r.lo, (double)(x >> 11) * 0x1p-53);
      worst = fmax(worst, ulp_error(f64_pow_full(t, r.c), powq(t, r.c)));
    }
    printf("%g..%g ^%.6f max_ulp=%.4f\n", r.lo, r.hi, r.c, worst);
  }
  for (double t : {1.0, 0.5, 2.0}) printf("%g ^0 max_ulp=%.4f\n", t, ulp_error(f64_pow_full(t, 0.0), 1.0Q));
  long differ = 0, n = 0;
  auto check = [&](double a, double c) {
    const double q = f64_div_by(a, c, 1.0 / c), r = a / c;
    differ += !(q == r || (q != q && r != r));
    n++;
  };
  auto uniform = [&]() {
    x ^= x << 13;
    x ^= x >> 7;
    x ^= x << 17;
    return (double)(x >> 11) * 0x1p-53;
  };
  const double inf = __builtin_inf(), nan = __builtin_nan("");
  for (int q = 0; q < 3000000; q++) {
    const double c = q % 3 == 0 ? 1e5 : q % 3 == 1 ? (double)(float)(0.5 + uniform()) * (double)(float)(0.5 + uniform()) : 0.5 + uniform();
    // a quotient near the middle between two doubles as often as not
    check(ldexp(1.0 + uniform(), (int)(uniform() * 200.0) - 100), c);
    check((1.0 + uniform()) * c * (1.0 + 0x1p-53 * (uniform() - 0.5)), c);
  }
  for (double a : {inf, -inf, nan, 0.0, -0.0, 1.5, -1e-30})
    for (double c : {1e5, -2.0, inf, -inf, 0.0, -0.0, nan}) check(a, c);
  printf("div checked=%ld differ=%ld\n", n, differ);
  return 0;
}
