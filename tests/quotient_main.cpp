// Counts the dividends of a range of exponents whose quotient by d (mh_div.h)
// differs from the IEEE division's: quotient_main d exponent_lo exponent_hi step
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "mh_div.h"

int main(int, char** argv) {
  const float d = std::strtof(argv[1], nullptr), inv = 1.0f / d;
  const int lo = std::atoi(argv[2]), hi = std::atoi(argv[3]);
  const uint32_t step = (uint32_t)std::atoi(argv[4]);
  unsigned long long bad = 0, n = 0;
  for (int e = lo; e <= hi; ++e)
    for (uint32_t sign = 0; sign < 2; ++sign)
      for (uint32_t m = 0; m < (1u << 23); m += step) {
        const uint32_t bits = (sign << 31) | ((uint32_t)(e + 127) << 23) | m;
        float a;
        std::memcpy(&a, &bits, 4);
        const float q = mh::quotient(a, d, inv), x = a / d;
        bad += std::memcmp(&q, &x, 4) != 0;
        ++n;
      }
  const float zero = mh::quotient(0.0f, d, inv);
  std::printf("%llu %llu %d\n", bad, n, zero == 0.0f);
}
