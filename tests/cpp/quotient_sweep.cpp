// Sweep of the two short quotients of the affine quantizer
// (mlx-llm_amd/csrc/affine_group.hpp) against the f32 division, on the CPU.
// The reciprocal estimate (v_rcp_f32, within one ulp) is tried as the nearest
// float to 1/n and as its two neighbours, so the result does not depend on
// how a device rounds it.
//   div   every mantissa of x, every odd n of 1 .. 257 (an even n is an odd
//         one at another exponent): fma(fma(-n, q, x), r, q) == x / n
//   rint  mantissas of s (every one below 16.5, every `step`-th above), every
//         half-integer h up to 256.5, the nine x around s h:
//         rint(fma(x, r1, x r2)) == rint(x / s) unless s has all mantissa bits
// Prints the number of differences of each and exits with 0 if there are none.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <thread>
#include <vector>

static float from_bits(uint32_t u) {
  float f;
  std::memcpy(&f, &u, 4);
  return f;
}
static uint32_t to_bits(float f) {
  uint32_t u;
  std::memcpy(&u, &f, 4);
  return u;
}
constexpr uint32_t kOne = 0x3F800000u, kMantissas = 1u << 23;

static int64_t div_range(int n_first, int n_step) {
  int64_t bad = 0;
  for (int ni = n_first; ni <= 257; ni += n_step) {
    const float n = static_cast<float>(ni);
    for (int e = -1; e <= 1; e++) {
      if (ni == 1 && e) continue;  // 1/1 is a float: its estimate is exact
      const float r = from_bits(to_bits(1.0f / n) + e);
      int32_t b = 0;
      for (uint32_t m = 0; m < kMantissas; m++) {
        const float x = from_bits(kOne | m);
        const float q = x * r;
        b += std::fmaf(std::fmaf(-n, q, x), r, q) != x / n;
      }
      bad += b;
    }
  }
  return bad;
}

static int64_t rint_range(uint32_t first, uint32_t threads, uint32_t step) {
  int64_t bad = 0;
  for (uint32_t m = first; m < kMantissas - 1; m += threads) {  // all ones: the quantizer divides
    const float s = from_bits(kOne | m);
    const int last = m % step == 0 ? 513 : 33;
    for (int e = -1; e <= 1; e++) {
      if (m == 0 && e) continue;
      const float r0 = from_bits(to_bits(1.0f / s) + e);
      const float r1 = std::fmaf(std::fmaf(-s, r0, 1.0f), r0, r0);
      const float r2 = std::fmaf(-s, r1, 1.0f) * r1;
      int32_t b = 0;
      for (int h2 = 1; h2 <= last; h2 += 2) {
        const uint32_t c = to_bits(s * (0.5f * static_cast<float>(h2)));
        for (int d = -4; d <= 4; d++) {
          const float x = from_bits(c + d);
          b += std::nearbyintf(std::fmaf(x, r1, x * r2)) != std::nearbyintf(x / s);
        }
      }
      bad += b;
    }
  }
  return bad;
}

int main() {
  const unsigned T = std::max(1u, std::min(16u, std::thread::hardware_concurrency()));
  std::vector<int64_t> div(T), rnt(T);
  std::vector<std::thread> pool;
  for (unsigned t = 0; t < T; t++)
    pool.emplace_back([&, t] {
      div[t] = div_range(1 + 2 * static_cast<int>(t), 2 * static_cast<int>(T));
      rnt[t] = rint_range(t, T, 61);
    });
  for (auto& p : pool) p.join();
  int64_t d = 0, r = 0;
  for (unsigned t = 0; t < T; t++) d += div[t], r += rnt[t];
  std::printf("div %lld rint %lld\n", static_cast<long long>(d), static_cast<long long>(r));
  return d || r;
}
