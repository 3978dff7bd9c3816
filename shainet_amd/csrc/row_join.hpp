// One row between two sublayers (residual_kernels.hpp) inside the launch that reads it next: every workgroup of 256 threads
// works it out for itself, from 44 KB at 1024 columns that come from the L2s while the product's own weights are on their
// way, and one of them leaves it for later launches.
#pragma once
#include "residual_kernels.hpp"

namespace shainet {

// XO: 16-byte pieces per thread, the row has 1024 XO columns; at most four taps.
template <int XO>
struct JoinRow {
  typedef float piece_t __attribute__((ext_vector_type(4)));
  piece_t x[XO], y[XO], post[XO], pre[XO], tap[XO][4], old[XO][3];

  // (something is requested in the place of what is not there: no load hangs on a condition)
  __device__ __forceinline__ void request(const ResidualArgs &a) {
    const piece_t *const xs = (const piece_t *)a.x, *const ys = (const piece_t *)(a.y ? a.y : a.x), *const ps = (const piece_t *)(a.y ? a.post : a.pre);
    const piece_t *const cs = (const piece_t *)(a.conv ? a.conv : a.pre), *const hs = (const piece_t *)(a.hist_in ? a.hist_in : a.pre);
#pragma unroll
    for (int i = 0; i < XO; ++i) {
      const int at = threadIdx.x + 256 * i;
      x[i] = xs[at];
      y[i] = ys[at];
      post[i] = ps[at];
      pre[i] = ((const piece_t *)a.pre)[at];
#pragma unroll
      for (int k = 0; k < 4; ++k) tap[i][k] = cs[(a.conv ? min(k, a.taps - 1) : 0) * 256 * XO + at];
#pragma unroll
      for (int k = 0; k < 3; ++k) old[i][k] = hs[(a.hist_in ? max(min(k, a.taps - 2), 0) : 0) * 256 * XO + at];
    }
  }

  // x becomes what the next sublayer reads.  red: LDS, a float per wavefront and sum; writes: whether this workgroup leaves
  // the joined row, the convolution's inputs and (a.h not null) the result.
  __device__ __forceinline__ void finish(const ResidualArgs &a, float (&red)[8], bool writes) {
    auto factor = [&](const piece_t (&v)[XO], float *r) {
      float sq = 0.f;
#pragma unroll
      for (int i = 0; i < XO; ++i) {
        const piece_t q = v[i] * v[i];
        sq += (q.x + q.y) + (q.z + q.w);
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) sq += __shfl_xor(sq, o);
      if ((threadIdx.x & 63) == 0) r[threadIdx.x >> 6] = sq;
      __syncthreads();
      return 1.0f / sqrtf((((r[0] + r[1]) + r[2]) + r[3]) / (float)(1024 * XO) + a.eps);
    };
    if (a.y) {
      const float f = factor(y, red);
#pragma unroll
      for (int i = 0; i < XO; ++i) {
        x[i] += y[i] * f * post[i];
        if (writes) ((piece_t *)a.x_out)[threadIdx.x + 256 * i] = x[i];
      }
    }
    const float f = factor(x, red + 4);
#pragma unroll
    for (int i = 0; i < XO; ++i) {
      const int at = threadIdx.x + 256 * i;
      const piece_t h = x[i] * f * pre[i];
      piece_t c = {0.f, 0.f, 0.f, 0.f};
      if (a.conv) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          if (k == a.taps - 1) c += h * tap[i][k];
          if (k < 3 && k < a.taps - 1) {
            const piece_t before = a.hist_in ? old[i][k] : piece_t{0.f, 0.f, 0.f, 0.f};
            c += before * tap[i][k];
            if (writes && a.hist_out && k > 0) ((piece_t *)a.hist_out)[(k - 1) * 256 * XO + at] = before;
          }
        }
        if (writes && a.hist_out && a.taps > 1) ((piece_t *)a.hist_out)[(a.taps - 2) * 256 * XO + at] = h;
      }
      x[i] = h + c;
      if (writes && a.h) ((piece_t *)a.h)[at] = x[i];
    }
  }
};

}  // namespace shainet
