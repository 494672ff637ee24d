// Host build of phlegethon_amd/csrc/phlx_fp64.hpp: the quotient and the square
// root with hardware seeds of any error up to their bound.
#include <cmath>
#include <cstdint>
#include <cstring>
#include <limits>

#include "../phlegethon_amd/csrc/phlx_fp64.hpp"

static double g_eps = 0.0;  // relative error of the seeds

namespace phlx {
double hw_rcp(double x) { return (1.0 / x) * (1.0 + g_eps); }
double hw_rsq(double x) { return (1.0 / std::sqrt(x)) * (1.0 + g_eps); }
double hw_div_fixup(double q, double b, double a) {
  const bool neg = std::signbit(a) != std::signbit(b);
  const double inf = std::numeric_limits<double>::infinity(), sg = neg ? -1.0 : 1.0;
  if (std::isnan(a) || std::isnan(b) || (a == 0.0 && b == 0.0) || (std::isinf(a) && std::isinf(b)))
    return std::numeric_limits<double>::quiet_NaN();
  if (b == 0.0 || std::isinf(a)) return sg * inf;
  if (std::isinf(b) || a == 0.0) return sg * 0.0;
  return std::copysign(q, sg);
}
}  // namespace phlx

using phlx::dsqrt;
using phlx::Recip;

static uint64_t g_s = 88172645463325252ull;
static uint64_t rnd() {
  g_s ^= g_s << 13;
  g_s ^= g_s >> 7;
  g_s ^= g_s << 17;
  return g_s * 0x2545F4914F6CDD1Dull;
}
static double make(uint64_t mant, int e) {
  const uint64_t u = ((uint64_t)(1023 + e) << 52) | (mant & 0xFFFFFFFFFFFFFull);
  double d;
  std::memcpy(&d, &u, 8);
  return d;
}
static const double kSeed = 0x1p-24;
static void random_seed_error() { g_eps = kSeed * ((double)(int64_t)rnd() * 0x1p-63); }
static long ulps(double a, double b) {
  int64_t x, y;
  std::memcpy(&x, &a, 8);
  std::memcpy(&y, &b, 8);
  return x > y ? x - y : y - x;
}

extern "C" void set_seed_error(double e) { g_eps = e; }
extern "C" double quotient(double a, double b) { return Recip(b).div(a); }
extern "C" double reciprocal(double b) { return Recip(b).inv(); }
extern "C" double root(double x) { return dsqrt(x); }

// n operands of exponents to +-300 (roots +-900): results that differ
extern "C" long random_mismatches(long n) {
  long bad = 0;
  for (long t = 0; t < n; t++) {
    random_seed_error();
    const uint64_t u = rnd(), v = rnd();
    double a = make(u, (int)(rnd() % 601) - 300);
    const double b = make(v, (int)(rnd() % 601) - 300);
    if (u >> 63) a = -a;
    const Recip r(b);
    const double x = make(v, (int)(rnd() % 1801) - 900);
    bad += (r.div(a) != a / b) + (r.inv() != 1.0 / b) + (dsqrt(x) != std::sqrt(x));
  }
  return bad;
}

// Quotients one unit of the exact product from a midpoint of two numbers, the
// closest there are: midpoint m (54 bits) = -+ 1/b mod 2^k, a = (m b +- 1) / 2^k.
// Largest distance from a / b in ulp; *count of them.
extern "C" long hardest_quotients(long n, long *count) {
  long worst = 0;
  *count = 0;
  for (long t = 0; t < n; t++) {
    uint64_t b = (1ull << 52) | (rnd() >> 12) | 1;
    if (t % 4 == 0) b = (1ull << 53) - 1 - 2 * (rnd() % 4096);
    if (t % 4 == 1) b = (1ull << 52) + 1 + 2 * (rnd() % 4096);
    uint64_t inv = b;
    for (int i = 0; i < 6; i++) inv *= 2 - b * inv;
    for (int sg = -1; sg <= 1; sg += 2)
      for (int k = 53; k <= 54; k++) {
        uint64_t m = (sg < 0 ? inv : 0 - inv) & ((1ull << k) - 1);
        if (k == 53) m |= 1ull << 53;
        if (m < (1ull << 53)) continue;
        unsigned __int128 p = (unsigned __int128)m * b;
        p = sg > 0 ? p + 1 : p - 1;
        if ((uint64_t)p & ((1ull << k) - 1)) continue;
        const uint64_t a = (uint64_t)(p >> k);
        if (a >> 53) continue;
        ++*count;
        random_seed_error();
        const long d = ulps(Recip((double)b).div((double)a), (double)a / (double)b);
        if (d > worst) worst = d;
      }
  }
  return worst;
}

// Roots as close to a midpoint: x 2^k = M^2 + M - c for small even c, M from the
// solution of M^2 + M = c mod 2^k lifted from mod 2.
extern "C" long hardest_roots(long *count) {
  long worst = 0;
  *count = 0;
  for (int k = 52; k <= 53; k++)
    for (int c = -1024; c <= 1024; c += 2)
      for (uint64_t m0 = 0; m0 < 2; m0++) {
        uint64_t M = m0;
        for (int i = 0; i < 7; i++) {
          const uint64_t f = M * M + M - (uint64_t)(int64_t)c, d = 2 * M + 1;
          uint64_t inv = d;
          for (int q = 0; q < 6; q++) inv *= 2 - d * inv;
          M -= f * inv;
        }
        M &= (1ull << k) - 1;
        if (k == 52) M |= 1ull << 52;
        if (M < (1ull << 52)) continue;
        const __int128 X = (__int128)M * M + M - c;
        if ((uint64_t)X & ((1ull << k) - 1)) continue;
        const uint64_t xi = (uint64_t)(X >> k);
        if ((uint64_t)(double)xi != xi) continue;
        const double x = std::ldexp((double)xi, k - 104);
        ++*count;
        for (int e = 0; e < 16; e++) {
          random_seed_error();
          const long d = ulps(dsqrt(x), std::sqrt(x));
          if (d > worst) worst = d;
        }
      }
  return worst;
}

// Operands whose remainder underflows: products of two slopes over their sum,
// and roots down to the smallest subnormal.  Largest distance in ulp.
extern "C" long smallest_operands(long n) {
  long worst = 0;
  for (long t = 0; t < n; t++) {
    random_seed_error();
    const double p = make(rnd(), -400 - (int)(rnd() % 138));
    const double q = make(rnd(), -400 - (int)(rnd() % 138));
    if (p * q > 0.0) {
      const long d = ulps(Recip(p + q).div(p * q), p * q / (p + q));
      if (d > worst) worst = d;
    }
    const double x = std::ldexp(make(rnd(), 0), -900 - (int)(rnd() % 175));
    if (x > 0.0) {
      const long d = ulps(dsqrt(x), std::sqrt(x));
      if (d > worst) worst = d;
    }
  }
  return worst;
}
