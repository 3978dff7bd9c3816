// A value of each lane and those of the lanes 16, 32 and 48 away, by register swaps: no trip to LDS.
#pragma once
#include <hip/hip_runtime.h>

namespace shainet {

template <typename F>
__device__ __forceinline__ float across_quarters(float x, F two) {
  auto both = [&](unsigned a, unsigned b) { return two(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b)); };
  unsigned bits = __builtin_bit_cast(unsigned, x);
  auto p = __builtin_amdgcn_permlane16_swap(bits, bits, false, false);
  bits = __builtin_bit_cast(unsigned, both(p[0], p[1]));
  p = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
  return both(p[0], p[1]);
}
__device__ __forceinline__ float max_across_quarters(float x) {
  return across_quarters(x, [](float a, float b) { return fmaxf(a, b); });
}
// (the same order in every lane but for the two sides of a sum)
__device__ __forceinline__ float sum_across_quarters(float x) {
  return across_quarters(x, [](float a, float b) { return a + b; });
}

// Quarter j's v[i] and quarter i's v[j] trade places.
__device__ __forceinline__ void trade_quarters(float &a, float &b, bool halves) {
  const unsigned x = __builtin_bit_cast(unsigned, a), y = __builtin_bit_cast(unsigned, b);
  auto p = halves ? __builtin_amdgcn_permlane32_swap(x, y, false, false) : __builtin_amdgcn_permlane16_swap(x, y, false, false);
  a = __builtin_bit_cast(float, (unsigned)p[0]);
  b = __builtin_bit_cast(float, (unsigned)p[1]);
}
template <typename V>
__device__ __forceinline__ void transpose_quarters(V (&v)[4]) {
#pragma unroll
  for (int halves = 1; halves >= 0; --halves)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const int first = halves ? i : 2 * i, second = halves ? i + 2 : 2 * i + 1;
        float a = v[first][w], b = v[second][w];
        trade_quarters(a, b, halves);
        v[first][w] = a;
        v[second][w] = b;
      }
}

}  // namespace shainet
