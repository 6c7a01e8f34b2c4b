// Exhaustive check of ConstDiv (cpml_constdiv.h) in float over every
// significand in a set of binades, and a random one in double.
// usage: const_div_check step   (every step-th significand; 1: all)
// Prints the number of quotients compared; exit code 1 at the first mismatch.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <initializer_list>

#include "../../seismic_cpml_amd/csrc/cpml_constdiv.h"

template <typename T, typename U>
static int check(const cpml::ConstDiv<T> &c, U bits) {
  T x;
  std::memcpy(&x, &bits, sizeof x);
  if (!c.in_range(x)) return 0;
  const T q = c.quot(x), r = x / c.d;
  if (std::memcmp(&q, &r, sizeof q) != 0) {
    std::printf("mismatch: %a / %a = %a, got %a\n", (double)x, (double)c.d, (double)r, (double)q);
    return -1;
  }
  return 1;
}

int main(int argc, char **argv) {
  const uint32_t step = argc > 1 ? (uint32_t)std::atoi(argv[1]) : 1;
  const double ds[] = {24, 5, 10, 120, 240, 36, 1.5, 4, 3, 7.3, 0.1, 0.0123, 1000, 24000, 1.9999999,
                       1.0000001, 0x1p-20, 1e12};
  long n = 0;
  uint64_t seed = 88172645463325252ull;
  for (double dd : ds) {
    const cpml::ConstDiv<float> c = cpml::const_div((float)dd);
    // exponents: subnormals and the smallest binades, the middle, the largest
    for (uint32_t e : {0u, 1u, 30u, 31u, 32u, 33u, 36u, 38u, 48u, 71u, 100u, 127u, 160u, 200u, 250u, 252u, 253u})
      for (uint32_t m = 0; m < (1u << 23); m += step)
        for (uint32_t sign : {0u, 1u}) {
          const int r = check(c, (sign << 31) | (e << 23) | m);
          if (r < 0) return 1;
          n += r;
        }
    const cpml::ConstDiv<double> cd = cpml::const_div(dd);
    for (int k = 0; k < 400000; ++k) {
      seed ^= seed << 13, seed ^= seed >> 7, seed ^= seed << 17;
      uint64_t b = seed;
      if (k % 4 == 0) b = (b & 0x800fffffffffffffull) | ((seed >> 20) % 60) << 52;  // tiny
      const int r = check(cd, b);
      if (r < 0) return 1;
      n += r;
    }
  }
  // what in_range must let through and what it must not
  const cpml::ConstDiv<float> c = cpml::const_div(24.f);
  const cpml::ConstDiv<double> cd = cpml::const_div(24.0);
  const double inf = HUGE_VAL;
  if (!c.in_range(0.f) || !c.in_range(-0.f) || !c.in_range(-1e-20f) || !c.in_range(1e30f) ||
      c.in_range(1e-40f) || c.in_range((float)inf) || !cd.in_range(0.0) || cd.in_range(5e-324) ||
      cd.in_range(-1e-300) || !cd.in_range(1e-200) || cd.in_range(-inf)) {
    std::printf("range test\n");
    return 1;
  }
  std::printf("%ld quotients equal\n", n);
  return 0;
}
