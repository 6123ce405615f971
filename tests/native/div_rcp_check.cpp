// fp::div_by_rcp(a, b, RN(1 / b)) against a / b, in two parts; prints the number of pairs checked and of bit
// mismatches of each.
//
// 1. Every pair that could be misrounded.  Scale a and b to [1, 2) and let x = a / b.  Each of the steps
//    y = RN(1 / b), q = RN(a y), r = RN(a - b q) has a relative error of at most 2^-24 (y's error is at most
//    2^-25 and b < 2), so |q - x| <= x (2^-23 + 2^-48), and the value that the last operation rounds,
//    q + r y = x + (x - q) (e_r + e_y + e_r e_y), is within x 2^-46 (1 + 2^-24)^2 of x.  It rounds as x does
//    unless a midpoint of two floats lies between them (x itself is none: a midpoint has 25 bits, and its
//    product with b would need 25).  With integer significands a = A / 2^23, b = B / 2^23 a midpoint is
//    M / 2^s with M odd in (2^24, 2^25), s = 24 for x >= 1 and 25 for x < 1, at the distance
//    |A 2^s - B M| / (B 2^s).  So K = A 2^s - B M is a non-zero integer with
//    |K| <= B 2^s x 2^-46 (1 + 2^-24)^2 = A 2^(s - 46) (1 + 2^-24)^2, at most 4 (s = 24) or 8 (s = 25).
//    For each B and K the solutions M of B M = -K (mod 2^s) give every such A.
// 2. Random pairs over the range of exponents that the callers allow.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>

#include "../../feriphys_amd/csrc/exact_ops.hpp"

namespace {

bool differs(float a, float b) {
  const float want = a / b, got = fp::div_by_rcp(a, b, 1.0f / b);
  return std::memcmp(&want, &got, 4) != 0;
}

uint64_t mix(uint64_t z) {
  z += 0x9e3779b97f4a7c15ull;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}

}  // namespace

int main() {
  unsigned long long pairs = 0, bad = 0, random_bad = 0;
  const long long lo = 1ll << 23, hi = 1ll << 24;
#pragma omp parallel for reduction(+ : pairs, bad) schedule(static)
  for (long long B = lo; B < hi; ++B) {
    const int t = __builtin_ctzll((unsigned long long)B);
    if (t > 3) continue;  // M is odd, so K has B's factors of two
    const uint64_t odd = (uint64_t)B >> t;
    uint64_t inv = odd;  // odd * inv = 1 (mod 2^64), by Newton's iteration
    for (int k = 0; k < 5; ++k) inv *= 2 - odd * inv;
    for (int s = 24; s <= 25; ++s)
      for (long long K = -(4 << (s - 24)); K <= (4 << (s - 24)); ++K) {
        if (K == 0 || K % (1ll << t) != 0) continue;
        const uint64_t step = 1ull << (s - t);
        for (uint64_t M = ((uint64_t)(-(K >> t)) * inv) & (step - 1); M < (1ull << 25); M += step) {
          if (M <= (1ull << 24) || M % 2 == 0) continue;
          const long long num = K + B * (long long)M;
          const long long A = num >> s;
          if (A * (1ll << s) != num) ++bad;  // M does not solve it
          if (A < lo || A >= hi || (s == 24) != (A >= B)) continue;
          ++pairs;
          bad += differs((float)A, (float)B) || differs(-(float)A, (float)B);
        }
      }
  }
  const long long n = 1ll << 27;
#pragma omp parallel for reduction(+ : random_bad) schedule(static)
  for (long long i = 0; i < n; ++i) {
    const uint64_t h = mix((uint64_t)i), g = mix(h);
    const float a = std::ldexp((float)((h & 0x7fffff) | 0x800000), (int)(g % 120) - 60 - 23);
    const float b = std::ldexp((float)((h >> 32 & 0x7fffff) | 0x800000), (int)(g / 120 % 120) - 60 - 23);
    random_bad += differs(g >> 40 & 1 ? -a : a, g >> 41 & 1 ? -b : b);
  }
  std::printf("%llu %llu %lld %llu\n", pairs, bad, n, random_bad);
  return 0;
}
