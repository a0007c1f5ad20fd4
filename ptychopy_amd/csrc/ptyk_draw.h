// Standard normal draws on the host, to the bit those of libstdc++'s std::normal_distribution<double> over
// std::mt19937_64 (the polar method: a pair of uniforms in the unit disc, two draws from it).
//
// Written out because the library's form asks for the two logarithms behind the number of words a uniform
// needs, in 80-bit arithmetic, for every draw: 37 or 66 ns each, depending on where the linker puts the
// code, which made the 1.94 M weights of a network take 70 or 128 ms (the whole network 74 or 132; now 19).
#pragma once
#include <cmath>
#include <cstdint>
#include <random>

namespace ptyk {

class NormalDraw {
 public:
  explicit NormalDraw(uint64_t seed) : g_(seed) {}
  double operator()() {
    if (have_) {
      have_ = false;
      return kept_;
    }
    double x, y, r;
    do {
      x = 2.0 * uniform() - 1.0;
      y = 2.0 * uniform() - 1.0;
      r = x * x + y * y;
    } while (r > 1.0 || r == 0.0);
    const double m = std::sqrt(-2.0 * std::log(r) / r);
    kept_ = x * m;
    have_ = true;
    return y * m;
  }

 private:
  double uniform() {  // [0, 1)
    const double u = (double)g_() * 0x1p-64;
    return u < 1.0 ? u : std::nextafter(1.0, 0.0);
  }
  std::mt19937_64 g_;
  double kept_ = 0.0;
  bool have_ = false;
};

}  // namespace ptyk
