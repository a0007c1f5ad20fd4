// NormalDraw gives the standard library's draws, bit for bit.
#include <cstdio>
#include <cstring>

#include "ptyk_draw.h"

int main() {
  for (uint64_t seed : {0ull, 1ull, 7ull, 12345ull, 0xffffffffffffffffull}) {
    std::mt19937_64 g(seed);
    std::normal_distribution<double> nd(0.0, 1.0);
    ptyk::NormalDraw d(seed);
    for (int i = 0; i < 1000000; ++i) {
      const double a = nd(g), b = d();
      if (std::memcmp(&a, &b, sizeof(a))) {
        std::printf("seed %llu draw %d: %.17g, not %.17g\n", (unsigned long long)seed, i, b, a);
        return 1;
      }
    }
  }
  return 0;
}
