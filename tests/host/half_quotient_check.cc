// The quotients of the binary16 softmax (mshadow/hip/kernels/softmax_half.h), checked exhaustively:
// for EVERY binary16 term in [0, 1] and EVERY binary16 sum in [1, 2048] the product with the sum's
// reciprocal as two floats is the float quotient bit for bit, and rounds to the binary16 number that
// half_t's `t / sum` (divided in float, rounded to nearest even) is. It also counts the pairs for
// which the exact product rounded once, straight to binary16, would be another number.
// Prints "OK <pairs> <pairs that one rounding would change>" and exits 0.
#include <immintrin.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>

static inline float Widen(uint16_t h) { return _cvtsh_ss(h); }
static inline uint16_t Narrow(float f) { return _cvtss_sh(f, _MM_FROUND_TO_NEAREST_INT); }
static inline uint32_t Bits(float f) {
  uint32_t u;
  std::memcpy(&u, &f, 4);
  return u;
}

int main() {
  unsigned long long pairs = 0, once = 0;
  for (uint32_t s = 0x3c00u; s <= 0x6800u; ++s) {
    const float sum = Widen(static_cast<uint16_t>(s));
    const float high = 1.0f / sum;
    const float low = std::fma(-sum, high, 1.0f) * high;
    for (uint32_t t = 0; t <= 0x3c00u; ++t) {
      const float term = Widen(static_cast<uint16_t>(t));
      const float small = term * low;
      const float p = std::fma(term, high, small);
      const float want = term / sum;
      if (Bits(p) != Bits(want) || Narrow(p) != Narrow(want)) {
        std::printf("FAIL term %04x sum %04x: %a, not %a\n", t, s, p, want);
        return 1;
      }
      // the exact value of term * high + small, truncated to a float whose last bit is set where
      // anything was cut off: that float rounds to binary16 as the exact value does
      const double product = static_cast<double>(term) * static_cast<double>(high);  // 11 and 24 bits: exact
      const double total = product + static_cast<double>(small);
      const double lost = (product - total) + static_cast<double>(small);
      float cut = static_cast<float>(total);
      if (static_cast<double>(cut) > total || (static_cast<double>(cut) == total && lost < 0.0)) {
        cut = std::nextafterf(cut, 0.0f);
      }
      if (static_cast<double>(cut) != total || lost != 0.0) {
        const uint32_t bits = Bits(cut) | 1u;
        std::memcpy(&cut, &bits, 4);
      }
      once += Narrow(cut) != Narrow(want) ? 1 : 0;
      ++pairs;
    }
  }
  std::printf("OK %llu %llu\n", pairs, once);
  return 0;
}
