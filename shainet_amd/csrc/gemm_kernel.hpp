// Launcher of the product y[T,N] = x[T,K] W[K,N] (+ res) for five rows and more, fp32 on the bf16 matrix cores.
#pragma once
#include <hip/hip_runtime.h>

#include "activation.hpp"

namespace shainet {

// What happens to y next, where a kernel of its own adds the pieces of a product's tiles (GemmPlan::pieces > 1).
struct NextNorm {
  int kind = 0;          // kNorm*
  const float *gamma = nullptr, *beta = nullptr;
  float alpha = 0.f;
  double eps = 0.0;
  float *rows = nullptr;  // [T, N]: the norm of y's rows goes there (null: none)
  bool planes = false;    // as their parts (split_mfma.hpp, store_planes); W of one part
};
struct GemvPrep;  // attn_kernels.hpp
struct GemmNext {
  NextNorm norm;
  const GemvPrep *prep = nullptr;  // N = q | k | v heads, without norms and biases: rotated and put where it says (y is not written)
  bool swiglu = false;  // N = gate | up, and y is [T, N / 2]: silu(gate) * up
};

struct GemmPlan {
  bool mfma;              // false: K, N or the row stride of x is not a multiple of 4 -> the plain kernel
  bool few;               // tiles of 32 rows and 128 columns, K steps of 32 (parts 1: see kg)
  int mb, wn;             // otherwise tiles of 64 mb rows and 64 wn columns, K steps of 16
  int kg;                 // few, parts 1: tiles of 32 mb rows and 256 / kg columns, K steps of 16 kg
  int tiles_m, tiles_n;
  int parts;              // bf16 numbers that a weight is the sum of: 3, or 1 where the weights are bf16 numbers
  int steps;              // K steps per tile; a unit of work is one step of one tile
  int group_bits;         // 2^group_bits groups of workgroups, each with an equal run of the tiles
  int tiles_per_group;
  int quota;              // consecutive units per workgroup (= steps: a workgroup per tile, nothing shared)
  int pieces;             // > 1: every tile is cut into this many pieces of `quota` steps and a second kernel adds them
  int workgroups;
  size_t partial_floats;  // scratch for the pieces of tiles that two or more workgroups share (0: none)
  size_t flag_words;      // words, zero before the first launch (the kernel leaves them zero), that mark pieces complete
};
// w_bf16: every value of W is a bf16 number
GemmPlan plan_gemm(int T, int K, int N, long long x_stride, bool w_bf16 = false);
void describe_gemm(const GemmPlan &p, int K, int plan[7]);  // shainet_hip_describe_matmul
// Device pointers, 16-byte aligned for the MFMA kernel; rows of x are x_stride floats apart, y and
// res are dense [T, N]; res nullable (y = res + x W; res == y is allowed);
// bias [N] nullable (y = act(x W + bias), before res is added).  partials, flags:
// p.partial_floats floats and p.flag_words words (unused when those are 0); error: a word the
// kernel sets to 1 when it gives up a wait for another workgroup's piece (y is invalid then).
// flag_set, spin_limit: for the test of the give-up path only (marks go to flag_set, p.flag_words
// words of their own, instead of flags, and a wait ends after spin_limit polls); null / 0 otherwise.
hipError_t launch_gemm(const float *x, long long x_stride, const float *w, float *y, const float *res, float *partials,
                       unsigned *flags, int *error, int T, int K, int N, const GemmPlan &p, hipStream_t stream,
                       unsigned *flag_set = nullptr, int spin_limit = 0, const float *bias = nullptr, Activation act = Activation(),
                       const GemmNext &next = GemmNext(), bool planes = false);
// planes: x is [3][T][K] of bf16, the parts of its lifted values (split_mfma.hpp, split_planes), in a product that takes it so.
bool gemm_takes_planes(const GemmPlan &p, int K);
// Whether the product's last launch does that, too.
bool gemm_takes_next(const GemmPlan &p, int T, int N, const GemmNext &next);

}  // namespace shainet
