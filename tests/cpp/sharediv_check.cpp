// Checks the branch-free quotients against IEEE division: DivBy (several
// quotients by one run-time divisor, from a reciprocal approximation with a
// relative error up to 2^-20) and div_unchecked (constant divisor) on the
// dividends that their range tests let through.
// usage: sharediv_check <n_random>; prints mismatches, exit 1 on any.
#include <cinttypes>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>

#include "../../sgn-hyperbolic-gpu_amd/csrc/sgnx_fastdiv.h"

static uint64_t bits(double x) { uint64_t u; std::memcpy(&u, &x, 8); return u; }
static double from_bits(uint64_t u) { double x; std::memcpy(&x, &u, 8); return x; }

static long bad = 0, tested = 0;
static void same(const char* what, double a, double b, double want, double got) {
  ++tested;
  if (bits(want) == bits(got)) return;
  if (bad++ < 10) std::printf("%s a=%a b=%a want=%a got=%a\n", what, a, b, want, got);
}

int main(int argc, char** argv) {
  const long n = argc > 1 ? std::atol(argv[1]) : 1000000;
  std::mt19937_64 rng(2024);
  std::uniform_real_distribution<double> U(-1.0, 1.0);
  auto random_mantissa = [&]() -> uint64_t {
    const uint64_t m = rng() & 0x000fffffffffffffULL;
    switch (rng() % 8) {                       // plain, and near the ends of the binade
      case 0: return m & 0xff;
      case 1: return 0x000fffffffffffffULL - (m & 0xff);
      case 2: return 0x000fffffffffffffULL - (m & 0xffffff);
      default: return m;
    }
  };
  auto divisor = [&](int range) {
    const uint64_t ex = 1023 - range + rng() % (2 * range);
    return from_bits(ex << 52 | random_mantissa());
  };
  auto dividend = [&]() {                      // 0, or 2^-900 <= |a| <= 2^800
    if (rng() % 64 == 0) return (rng() & 1) ? 0.0 : -0.0;
    const uint64_t ex = rng() % 4 ? 1023 - 60 + rng() % 120 : 1023 - 900 + rng() % 1700;
    return from_bits((rng() & 0x8000000000000000ULL) | ex << 52 | random_mantissa());
  };
  for (long i = 0; i < n; ++i) {
    const double b = divisor(100);
    const bool ones = (bits(b) & 0xffffffffULL) == 0xffffffffULL;   // left to IEEE division
    if (sgnx::div_by_ok(b) == ones) { ++bad; std::printf("div_by_ok(%a)\n", b); }
    if (ones) continue;
    const double y0 = (1.0 / b) * (1.0 + 0x1p-20 * U(rng));
    const sgnx::DivBy d = sgnx::make_div_by(b, y0);
    for (int k = 0; k < 4; ++k) {
      const double a = dividend();
      same("DivBy", a, b, a / b, d.quotient(a));
    }
    // neighbours of products and of half-way products of b
    const double m = from_bits((1023 + rng() % 40) << 52 | random_mantissa());
    for (double a : {m * b, std::nextafter(m * b, INFINITY), std::nextafter(m * b, 0.0),
                     (m + std::ldexp(m, -53)) * b})
      same("DivBy", a, b, a / b, d.quotient(a));
  }
  for (double b : {0.0, -1.0, 0x1p-101, 0x1p+100, (double)INFINITY, (double)NAN, -(double)INFINITY})
    if (sgnx::div_by_ok(b)) { ++bad; std::printf("div_by_ok(%a)\n", b); }
  for (double b : {0x1p-100, 0x1.ffffffffffffep+99, 1.0, 0x1.ffffffffffffep-1})
    if (!sgnx::div_by_ok(b)) { ++bad; std::printf("!div_by_ok(%a)\n", b); }
  // constant divisors: whatever the test and a finite result let through is a / b,
  // with +0 for either zero
  for (long i = 0; i < n / 100; ++i) {
    const double b = i < 50 ? std::ldexp(0x1.fffffffffffffp-1, (int)i - 25) : divisor(i % 2 ? 12 : 100);
    const sgnx::ConstDiv d = sgnx::make_const_div(b);
    for (int k = 0; k < 100; ++k) {
      double a = k % 2 ? from_bits(rng()) : dividend();
      if (k < 25 && k % 4 == 3) a = std::ldexp(1.0, k - 12);
      if (k == 0) a = from_bits((rng() & 0x8000000000000000ULL) | (rng() & 0x000fffffffffffffULL));
      if (sgnx::div_needs_exact(a) != (std::fabs(a) < 0x1p-900 && a != 0.0)) {
        ++bad;
        std::printf("div_needs_exact(%a)\n", a);
      }
      const double q = sgnx::div_unchecked(a, d);
      if (!sgnx::div_needs_exact(a) && std::isfinite(q)) same("unchecked", a, b, (a + 0.0) / b, q);
    }
  }
  std::printf("sharediv: %ld tested, %ld mismatches\n", tested, bad);
  return bad ? 1 : 0;
}
