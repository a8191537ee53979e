// The kernels' short quotient and square root (csrc/short_ops.inc) against the operators, on the CPU:
// the hardware's approximations 1/q and x^(-1/2) are replaced by the correctly rounded values times
// 1 + d, |d| <= 2^-22, d random or one of the ends (0 for a divisor with all mantissa bits set).
// Prints the number of results that differ.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#define __device__
#define __forceinline__ inline
static uint64_t state = 88172645463325252ull;
static uint64_t bits() {
  state ^= state << 13;
  state ^= state >> 7;
  state ^= state << 17;
  return state;
}
static double off() {                        // in [-2^-22, 2^-22]
  const uint64_t b = bits();
  if ((b & 7) == 0) return 0x1p-22;
  if ((b & 7) == 1) return -0x1p-22;
  return ((double)(int64_t)bits()) * 0x1p-63 * 0x1p-22;
}
static bool all_ones(double q) {
  uint64_t u;
  std::memcpy(&u, &q, 8);
  return (~u & 0xfffffffffffffull) == 0;
}
static double approx_rcp(double q) {
  return all_ones(q) ? 1.0 / q : (1.0 / q) * (1.0 + off());
}
static double approx_rsq(double x) { return (1.0 / std::sqrt(x)) * (1.0 + off()); }
#define __builtin_amdgcn_rcp approx_rcp
#define __builtin_amdgcn_rsq approx_rsq
using std::fma;
#include "short_ops.inc"

static double with_exponent(uint64_t mantissa, int e, bool negative) {
  uint64_t u = ((uint64_t)(e + 1023) << 52) | (mantissa & 0xfffffffffffffull) | (negative ? 1ull << 63 : 0);
  double d;
  std::memcpy(&d, &u, 8);
  return d;
}
static uint64_t mantissa() {                 // random, or within a few units of a power of two
  const uint64_t b = bits();
  if ((b & 3) == 0) return bits() % 5;
  if ((b & 3) == 1) return 0xfffffffffffffull - bits() % 5;
  return bits();
}
static int exponent(int lim) { return (int)(bits() % (2 * lim)) - lim; }

int main() {
  long bad = 0;
  auto quotient = [&](double e, double q) {
    if (e != 0.0 && (std::fabs(e) < 0x1p-400 || std::fabs(e) >= 0x1p400)) return;
    if (std::fabs(q) < 0x1p-400 || std::fabs(q) >= 0x1p400) return;
    const double want = e / q, got = short_quotient(e, q);
    if (want != got && bad++ < 5) std::printf("%a / %a: %a, not %a\n", e, q, got, want);
  };
  auto root = [&](double x) {
    if (x < 0x1p-400 || x >= 0x1p400) return;
    const double want = std::sqrt(x), got = short_sqrt(x);
    if (want != got && bad++ < 5) std::printf("sqrt %a: %a, not %a\n", x, got, want);
  };
  for (long i = 0; i < 6000000; ++i) {
    const double q = with_exponent(mantissa(), exponent(400), bits() & 1);
    quotient(with_exponent(mantissa(), exponent(400), bits() & 1), q);
    if ((i & 1023) == 0) quotient(0.0, q);
    // quotients near the middle between two doubles: e about q (t + half an ulp of t)
    const double t = with_exponent(bits(), exponent(100), false), h = std::ldexp(1.0, std::ilogb(t) - 53);
    const double s = with_exponent(bits(), exponent(250), bits() & 1), e = std::fma(s, h, s * t);
    quotient(e, s);
    quotient(std::nextafter(e, INFINITY), s);
    quotient(std::nextafter(e, -INFINITY), s);
    root(with_exponent(mantissa(), exponent(400), false));
    // roots near the middle: x about (t + half an ulp)^2
    const double x = std::fma(2.0 * t, h, t * t);
    root(x);
    root(std::nextafter(x, INFINITY));
    root(std::nextafter(x, 0.0));
  }
  std::printf("%ld\n", bad);
  return bad != 0;
}
