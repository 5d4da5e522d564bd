// substep_helpers_main.cpp — CPU check of FastDiv (phasefield_amd/csrc/pf_diffuse_direct.h): quotient
// and remainder against the division for divisors and dividends around every power of two and at
// random, up to 2^31 - 1.  tests/test_substep_helpers.py builds it with hipcc (host code) and runs it.
#include <cstdint>
#include <cstdio>
#include <random>
#include <vector>

#include "../phasefield_amd/csrc/pf_diffuse_direct.h"

int main() {
  std::vector<uint32_t> v;
  for (int b = 0; b < 31; ++b)
    for (int d = -2; d <= 2; ++d) {
      const int64_t x = (int64_t(1) << b) + d;
      if (x >= 1 && x <= 2147483647) v.push_back(uint32_t(x));
    }
  v.push_back(2147483647u);
  std::mt19937 rng(7);
  for (int q = 0; q < 300; ++q) v.push_back(1u + (rng() & 0x7fffffffu) % 2147483647u);
  for (int q = 0; q < 300; ++q) v.push_back(1u + rng() % 5000u);
  for (uint32_t d : v) {
    const pfamd::FastDiv f(d);
    auto ok = [&](uint32_t n) { return f.quot(n) == n / d && f.rem(n) == n % d; };
    bool good = ok(0);
    for (uint32_t n : v) {
      good = good && ok(n);
      const uint32_t m = n / d * d;  // the last multiple of d up to n, and the one before it
      good = good && ok(m) && (m == 0 || ok(m - 1));
    }
    if (!good) {
      std::fprintf(stderr, "FastDiv(%u) is wrong\n", d);
      return 1;
    }
  }
  std::printf("substep_helpers_main: ok\n");
  return 0;
}
