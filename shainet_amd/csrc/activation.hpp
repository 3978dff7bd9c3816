// Activations that ride in a product's epilogue, with their constants as parameters.
#pragma once
#include <hip/hip_runtime.h>

namespace shainet {

enum { kActNone = 0, kActXielu = 1 };
// kActXielu: pos z^2 + z / 2 for z > 0, neg (exp(z) - 1 - z) + z / 2 otherwise
struct Activation {
  int kind = kActNone;
  float pos = 0.f, neg = 0.f;
};

__device__ __forceinline__ float activate(const Activation &a, float z) {
  if (a.kind == kActXielu) return (z > 0.f ? a.pos * z * z : a.neg * (expm1f(z) - z)) + 0.5f * z;
  return z;
}

// silu(gate) up in fp64 (swiglu_ff.cr:84-89).  2^n times a series for the rest, up to 2^-47 of its value, and a reciprocal refined once to
// 2^-45: rounded to fp32 the same as the library's exp and a division, in a third of their instructions, which were most of what a
// launch of them took (512 rows of 2 x 8192 10.6 us).  Infinities and NaN as there.
__device__ __forceinline__ float swiglu(float gate, float up) {
  const double g = (double)gate, z = g * -1.4426950408889634;
  const double t = fmin(fmax(z, -1100.0), 1000.0), n = rint(t), r = (t - n) * 0.6931471805599453;
  double p = 1.0 / 39916800;
  p = fma(p, r, 1.0 / 3628800);
  p = fma(p, r, 1.0 / 362880);
  p = fma(p, r, 1.0 / 40320);
  p = fma(p, r, 1.0 / 5040);
  p = fma(p, r, 1.0 / 720);
  p = fma(p, r, 1.0 / 120);
  p = fma(p, r, 1.0 / 24);
  p = fma(p, r, 1.0 / 6);
  p = fma(p, r, 0.5);
  p = fma(p, r, 1.0);
  p = fma(p, r, 1.0);
  const double d = 1.0 + ldexp(p, (int)n);
  double q = __builtin_amdgcn_rcp(d);
  q = fma(fma(-d, q, 1.0), q, q);
  return (float)((z >= 1024.0 ? g * 0.0 : g * q) * (double)up);
}

}  // namespace shainet
