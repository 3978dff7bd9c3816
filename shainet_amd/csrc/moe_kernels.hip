// A mixture of experts on gfx950 (moe_kernels.hpp says what is computed), fp32.
#include "moe_kernels.hpp"
#include "row_join.hpp"
#include "split_mfma.hpp"

#include <math.h>
#include <stdint.h>
#include <stdlib.h>

namespace shainet {

namespace {

__device__ __forceinline__ float swiglu1(float g, float u) { return g / (1.f + expf(-g)) * u; }
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// The largest of v over the wavefront and, among equal ones, the smallest index.
__device__ __forceinline__ void wave_best(float &v, int &i) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float ov = __shfl_xor(v, o);
    const int oi = __shfl_xor(i, o);
    if (ov > v || (ov == v && oi < i)) {
      v = ov;
      i = oi;
    }
  }
}

// One wavefront chooses for one token.  logits: [n] (global); s, c: n floats of LDS each, best: m.groups floats
// of LDS.  ids, weights: m.top entries each, written by lane 0 (LDS or global).
__device__ __forceinline__ void choose(const MoeShape &m, const float *logits, const float *correction, float *s, float *c,
                                       float *best, int *ids, float *weights) {
  const int n = m.experts + m.identity, lane = threadIdx.x & 63, per = n / m.groups;
  if (n <= 64) {
    // a lane per output: who comes before whom is counted instead of searched for round by round
    const bool in = lane < n;
    const float z = in ? logits[lane] : -INFINITY, corr = in ? correction[lane] : 0.f;
    float top_z = z;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) top_z = fmaxf(top_z, __shfl_xor(top_z, o));
    const float e = in ? expf(z - top_z) : 0.f;
    const float p = e / wave_sum(e), x = p + corr;
    bool open = in;
    if (m.groups > 1) {
      if (in) c[lane] = x;
      __threadfence_block();
      const int mine = (in ? lane : 0) / per;
      float gb = -INFINITY;
#pragma unroll 4
      for (int i = 0; i < per; ++i) gb = fmaxf(gb, c[mine * per + i]);
      if (in && lane == mine * per) best[mine] = gb;
      __threadfence_block();
      int before = 0;
#pragma unroll 4
      for (int g = 0; g < m.groups; ++g) {
        const float v = best[g];
        before += v > gb || (v == gb && g < mine) ? 1 : 0;
      }
      open = in && before < m.keep;
    }
    if (in) s[lane] = open ? x : -INFINITY;
    __threadfence_block();
    int before = 0;
#pragma unroll 8
    for (int k = 0; k < n; ++k) {
      const float v = s[k];
      before += v > x || (v == x && k < lane) ? 1 : 0;
    }
    const bool chosen = open && before < m.top;
    const float total = wave_sum(chosen ? p : 0.f);
    for (int k = lane; k < m.top; k += 64) {  // (only with logits that are no numbers would an entry stay like this)
      ids[k] = 0;
      weights[k] = 0.f;
    }
    __threadfence_block();
    if (chosen) {
      ids[before] = lane;
      weights[before] = p / (total + 1e-20f) * m.scale;
    }
    __threadfence_block();
    return;
  }
  float mx = -INFINITY;
  for (int i = lane; i < n; i += 64) mx = fmaxf(mx, logits[i]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  float sum = 0.f;
  for (int i = lane; i < n; i += 64) {
    const float e = expf(logits[i] - mx);
    s[i] = e;
    sum += e;
  }
  sum = wave_sum(sum);
  for (int i = lane; i < n; i += 64) {
    const float p = s[i] / sum;
    s[i] = p;
    c[i] = p + correction[i];
  }
  __builtin_amdgcn_wave_barrier();
  __threadfence_block();
  if (m.groups > 1) {
    for (int g = lane; g < m.groups; g += 64) {
      float b = -INFINITY;
      for (int i = 0; i < per; ++i) b = fmaxf(b, c[g * per + i]);
      best[g] = b;
    }
    __threadfence_block();
    for (int k = 0; k < m.keep; ++k) {  // a kept group's entry becomes NaN: no comparison takes it again
      float v = -INFINITY;
      int at = 0x7fffffff;
      for (int g = lane; g < m.groups; g += 64) {
        const float b = best[g];
        if (b > v || (b == v && g < at)) {
          v = b;
          at = g;
        }
      }
      wave_best(v, at);
      if (at < m.groups && lane == 0) best[at] = NAN;
      __threadfence_block();
    }
    for (int i = lane; i < n; i += 64) {
      const float b = best[i / per];
      if (b == b) c[i] = NAN;
    }
    __threadfence_block();
  }
  float total = 0.f;
  for (int k = 0; k < m.top; ++k) {
    float v = -INFINITY;
    int at = 0x7fffffff;
    for (int i = lane; i < n; i += 64) {
      const float x = c[i];
      if (x > v || (x == v && i < at)) {
        v = x;
        at = i;
      }
    }
    wave_best(v, at);
    at = min(at, n - 1);  // (only with logits that are no numbers)
    const float p = s[at];
    total += p;
    if (lane == 0) {
      ids[k] = at;
      weights[k] = p;
      c[at] = NAN;
    }
    __threadfence_block();
  }
  for (int k = lane; k < m.top; k += 64) weights[k] = weights[k] / (total + 1e-20f) * m.scale;
  __threadfence_block();
}

// ---- a few tokens ------------------------------------------------------------------------------
// this lane's share of a . b, n floats
template <bool VEC>
__device__ __forceinline__ float dot_lane(const float *a, const float *b, int n) {
  const int lane = threadIdx.x & 63;
  float s = 0.f;
  if constexpr (VEC) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    const int n4 = n >> 2;
    int i = lane;
    for (; i + 192 < n4; i += 256) {
      f32x4 x[4], y[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        x[u] = __builtin_nontemporal_load((const f32x4 *)a + i + 64 * u);
        y[u] = ((const f32x4 *)b)[i + 64 * u];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) acc += x[u] * y[u];
    }
    for (; i < n4; i += 64) acc += ((const f32x4 *)a)[i] * ((const f32x4 *)b)[i];
    s = (acc.x + acc.y) + (acc.z + acc.w);
  } else {
    for (int i = lane; i < n; i += 64) s += a[i] * b[i];
  }
  return s;
}

// The same of one row that is still to be made (row_join.hpp): the first workgroup leaves it for the launches behind this
// one.  2.9 us and 3.9 for the row by itself; this way 4.2.
template <int XO>
__global__ __launch_bounds__(256) void moe_join_logits_kernel(const ResidualArgs join, const float *__restrict__ router, float *__restrict__ logits, int n) {
  constexpr int D = 1024 * XO;
  __shared__ __attribute__((aligned(16))) float xs[D];
  __shared__ float red[8];
  const int lane = threadIdx.x & 63, i = blockIdx.x * 4 + (threadIdx.x >> 6);
  JoinRow<XO> row;
  row.request(join);
  f32x4 w[4 * XO];
#pragma unroll
  for (int k = 0; k < 4 * XO; ++k) w[k] = *(const f32x4 *)(router + (long long)min(i, n - 1) * D + 256 * k + 4 * lane);
  row.finish(join, red, blockIdx.x == 0);
#pragma unroll
  for (int k = 0; k < XO; ++k) *(f32x4 *)(xs + 4 * threadIdx.x + 1024 * k) = row.x[k];
  __syncthreads();
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < 4 * XO; ++k) acc += w[k] * *(const f32x4 *)(xs + 256 * k + 4 * lane);
  const float s = wave_sum((acc.x + acc.y) + (acc.z + acc.w));
  if (lane == 0 && i < n) logits[i] = s;
}

// logits[t][n] = router row n . h row t: a wavefront each
template <bool VEC>
__global__ __launch_bounds__(256) void moe_logits_kernel(const float *__restrict__ h, const float *__restrict__ router,
                                                         float *__restrict__ logits, int n, int d) {
  const int i = blockIdx.x * 4 + (threadIdx.x >> 6), t = blockIdx.y;
  if (i >= n) return;
  const float s = wave_sum(dot_lane<VEC>(router + (long long)i * d, h + (long long)t * d, d));
  if ((threadIdx.x & 63) == 0) logits[(long long)t * n + i] = s;
}

// hidden[t][slot][j] = silu(gate row j . h) * (up row j . h) of the slot's expert; slot `top` is the shared one.
// A wavefront per output; blockIdx.x: the shared expert's outputs, then slot 0's, slot 1's ...  Every workgroup
// of a slot works the choice out again from the logits (a launch of its own would take longer) with one
// wavefront while the others bring h into LDS; the first one leaves it for moe_down_kernel.
template <bool VEC>
__global__ __launch_bounds__(256) void moe_up_kernel(MoeShape m, MoeTensors w, const float *__restrict__ h,
                                                     const float *__restrict__ logits, float *__restrict__ hidden,
                                                     int width, int shared_blocks, int slot_blocks,
                                                     int *__restrict__ ids_out, float *__restrict__ weights_out) {
  extern __shared__ __attribute__((aligned(16))) float smem[];  // h, s, c, best, weights, ids
  const int n = m.experts + m.identity, t = blockIdx.y;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const bool shared = (int)blockIdx.x < shared_blocks;
  const int slot = shared ? m.top : ((int)blockIdx.x - shared_blocks) / slot_blocks;
  const int j = (shared ? (int)blockIdx.x : ((int)blockIdx.x - shared_blocks) - slot * slot_blocks) * 4 + wave;
  const int ff = shared ? m.shared_ff : m.ff;
  const float *row = h + (long long)t * m.d;
  float *xs = smem;
  if (wave > 0) {
    if constexpr (VEC) {
      for (int i = threadIdx.x - 64; i < m.d >> 2; i += 192) ((f32x4 *)xs)[i] = ((const f32x4 *)row)[i];
    } else {
      for (int i = threadIdx.x - 64; i < m.d; i += 192) xs[i] = row[i];
    }
  } else if (shared) {
    // (nothing to choose)
  } else {
    float *s = smem + (m.d + 3) / 4 * 4, *weights = s + 2 * n + m.groups;
    int *ids = (int *)(weights + m.top);
    choose(m, logits + (long long)t * n, w.correction, s, s + n, s + 2 * n, ids, weights);
    if (slot == 0 && j == 0)
      for (int k = lane; k < m.top; k += 64) {
        ids_out[t * m.top + k] = ids[k];
        weights_out[t * m.top + k] = weights[k];
      }
  }
  __syncthreads();
  const float *gate = w.shared_gate_up;
  if (!shared) {
    const int e = ((const int *)(smem + (m.d + 3) / 4 * 4 + 2 * n + m.groups + m.top))[slot];
    if (e >= m.experts) return;
    gate = w.gate_up + (long long)e * 2 * m.ff * m.d;
  }
  if (j >= ff) return;
  float g, u;
  if constexpr (VEC) {  // both rows in flight together
    const f32x4 *gp = (const f32x4 *)(gate + (long long)j * m.d), *up = (const f32x4 *)(gate + (long long)(ff + j) * m.d);
    f32x4 ga = {0.f, 0.f, 0.f, 0.f}, ua = ga;
    const int n4 = m.d >> 2;
    constexpr int U = 8;
    for (int i0 = lane; i0 < n4; i0 += 64 * U) {
      f32x4 gv[U], uv[U];
#pragma unroll
      for (int k = 0; k < U; ++k)
        if (i0 - lane + 64 * k < n4) {
          const int i = min(i0 + 64 * k, n4 - 1);
          gv[k] = __builtin_nontemporal_load(gp + i);
          uv[k] = __builtin_nontemporal_load(up + i);
        }
#pragma unroll
      for (int k = 0; k < U; ++k)
        if (i0 + 64 * k < n4) {
          const f32x4 x = ((const f32x4 *)xs)[i0 + 64 * k];
          ga += gv[k] * x;
          ua += uv[k] * x;
        }
    }
    g = (ga.x + ga.y) + (ga.z + ga.w);
    u = (ua.x + ua.y) + (ua.z + ua.w);
  } else {
    g = dot_lane<false>(gate + (long long)j * m.d, xs, m.d);
    u = dot_lane<false>(gate + (long long)(ff + j) * m.d, xs, m.d);
  }
  g = wave_sum(g);
  u = wave_sum(u);
  if (lane == 0) hidden[((long long)t * (m.top + 1) + slot) * width + j] = swiglu1(g, u);
}

// y[t][j]: a wavefront per output, over all slots, four experts' rows in flight together
template <bool VEC>
__global__ __launch_bounds__(256) void moe_down_kernel(MoeShape m, MoeTensors w, const float *__restrict__ h,
                                                       const float *__restrict__ hidden, int width,
                                                       const int *__restrict__ ids, const float *__restrict__ weights,
                                                       float *__restrict__ y) {
  const int j = blockIdx.x * 4 + (threadIdx.x >> 6), t = blockIdx.y, lane = threadIdx.x & 63;
  if (j >= m.d) return;
  const float *hid = hidden + (long long)t * (m.top + 1) * width;
  float s = 0.f, same = 0.f;
  if constexpr (VEC) {
    constexpr int G = 4, U = 4;
    const int n4 = m.ff >> 2, s4 = m.shared_ff >> 2;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    if (m.shared_ff) {
      const f32x4 *a = (const f32x4 *)(w.shared_down + (long long)j * m.shared_ff), *b = (const f32x4 *)(hid + (long long)m.top * width);
      for (int i0 = 0; i0 < s4; i0 += 64 * 8) {
        f32x4 x[8], v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k)
          if (i0 + 64 * k < s4) {
            const int i = min(i0 + 64 * k + lane, s4 - 1);
            x[k] = __builtin_nontemporal_load(a + i);
            v[k] = b[i];
          }
#pragma unroll
        for (int k = 0; k < 8; ++k)
          if (i0 + 64 * k + lane < s4) acc += x[k] * v[k];
      }
    }
    for (int k0 = 0; k0 < m.top; k0 += G) {
      const f32x4 *a[G], *b[G];
      float wk[G];
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const int k = min(k0 + g, m.top - 1), e = ids[t * m.top + k];
        const bool real = k0 + g < m.top && e < m.experts;
        wk[g] = real ? weights[t * m.top + k] : 0.f;
        if (k0 + g < m.top && e >= m.experts) same += weights[t * m.top + k];
        a[g] = real ? (const f32x4 *)(w.down + ((long long)e * m.d + j) * m.ff) : nullptr;
        b[g] = (const f32x4 *)(hid + (long long)k * width);
      }
      for (int i0 = 0; i0 < n4; i0 += 64 * U) {
        f32x4 x[G][U], v[G][U];
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
          for (int u = 0; u < U; ++u)
            if (a[g] && i0 + 64 * u < n4) {
              const int i = min(i0 + 64 * u + lane, n4 - 1);
              x[g][u] = __builtin_nontemporal_load(a[g] + i);
              v[g][u] = b[g][i];
            }
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
          for (int u = 0; u < U; ++u)
            if (a[g] && i0 + 64 * u + lane < n4) acc += wk[g] * (x[g][u] * v[g][u]);
      }
    }
    s = (acc.x + acc.y) + (acc.z + acc.w);
  } else {
    for (int k = 0; k < m.top; ++k) {
      const int e = ids[t * m.top + k];
      const float wk = weights[t * m.top + k];
      if (e >= m.experts)
        same += wk;
      else
        s += wk * dot_lane<false>(w.down + ((long long)e * m.d + j) * m.ff, hid + (long long)k * width, m.ff);
    }
    if (m.shared_ff) s += dot_lane<false>(w.shared_down + (long long)j * m.shared_ff, hid + (long long)m.top * width, m.shared_ff);
  }
  s = wave_sum(s);
  if (lane == 0) y[(long long)t * m.d + j] = s + same * h[(long long)t * m.d + j];
}

// The same for at most G slots and experts of at most 256 U values, a multiple of 4: all rows, the shared expert's first
// 1024 values too, are requested before the first is looked at, where the kernel above goes to memory once per four slots and
// once for the shared expert (a launch is a wavefront per SIMD, and so these round trips; the same sums in the same
// order).  No load hangs on a condition: a slot without an expert's row has a buffer without records, whose loads come
// back as zeros and go nowhere.  (With branches around them the compiler had U = 1 wait for one load after the other, in 424
// registers: 18.6 us where it is 5.2 now.)  Two, four and eight slots, because such loads take their turn, too: 8 rows with 2
// slots of 768 10 us, in eight slots 19.  U = 3 holds 224 registers of rows in eight slots; a fourth span would not leave two
// wavefronts a SIMD, which several rows live on.
// One row | 8 rows, the kernel above -> this (us; 24 experts; slots x values -> outputs, shared values):
//   6 x 512 -> 1024, 1024  11.4 -> 5.3 | 30 -> 18.5      8 x 256 -> 1024, 512  9.2 -> 4.5 | 24 -> 12
//   8 x 768 -> 2048, 2048  19.9 -> 13.8 | 109 -> 77      8 x 256 -> 2048, none 9.0 -> 5.2 | 42 -> 21
//   8 x 512 -> 2048, 1024  14.7 -> 8.1 | 76 -> 43        4 x 768 -> 2048, none 10.1 -> 6.3 | 49 -> 31
//   2 x 768 -> 1024, none  6.4 -> 3.8 | 15.5 -> 9.8      1 x 256 -> 1024, none 3.9 -> 3.4 | 7.6 -> 5.9
template <int U, int G>
__global__ __launch_bounds__(256) void moe_down_once_kernel(MoeShape m, MoeTensors w, const float *__restrict__ h,
                                                            const float *__restrict__ hidden, int width,
                                                            const int *__restrict__ ids, const float *__restrict__ weights,
                                                            float *__restrict__ y) {
  constexpr int S = 4;
  const int j = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), t = blockIdx.y, lane = threadIdx.x & 63;
  if (j >= m.d) return;
  const float *hid = hidden + (long long)t * (m.top + 1) * width;
  const int n4 = m.ff >> 2, s4 = m.shared_ff >> 2;
  // piece i of a row of n (nothing is read beyond the row)
  auto row = [](const float *p, int n) { return __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, n * 4, 0x00027000); };
  auto piece = [](__amdgpu_buffer_rsrc_t r, int i) { return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, 16 * i, 0, 0)); };
  auto piece_once = [](__amdgpu_buffer_rsrc_t r, int i) { return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, 16 * i, 0, 2)); };
  const float *sa = w.shared_down + (long long)j * m.shared_ff, *sb = hid + (long long)m.top * width;
  // (the slots' experts and weights in lanes: as scalars they came one after the other, too)
  const int slot = t * m.top + min(lane, m.top - 1);
  const int id = lane < m.top ? ids[slot] : m.experts;
  const float weight = lane < m.top ? weights[slot] : 0.f;
  f32x4 x[G][U], v[G][U], sx[S], sv[S];
  const auto shared_w = row(sa, min(m.shared_ff, 256 * S)), shared_h = row(sb, min(m.shared_ff, 256 * S));
#pragma unroll
  for (int k = 0; k < S; ++k) {
    sx[k] = piece_once(shared_w, 64 * k + lane);
    sv[k] = piece(shared_h, 64 * k + lane);
  }
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int e = __builtin_amdgcn_readlane(id, g);
    const bool real = e < m.experts;
    const auto down = row(w.down + ((long long)(real ? e : 0) * m.d + j) * m.ff, real ? m.ff : 0), of = row(hid + (long long)g * width, real ? m.ff : 0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      x[g][u] = piece_once(down, 64 * u + lane);
      v[g][u] = piece(of, 64 * u + lane);
    }
  }
  __builtin_amdgcn_sched_barrier(0);  // (no sum starts, and waits, in front of the last load)
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < S; ++k) acc += sx[k] * sv[k];
  for (int i = 64 * S + lane; i < s4; i += 64) acc += __builtin_nontemporal_load((const f32x4 *)sa + i) * ((const f32x4 *)sb)[i];
  float same = 0.f;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const bool real = __builtin_amdgcn_readlane(id, g) < m.experts;
    const float wk = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, weight), g));
    same += real ? 0.f : wk;
#pragma unroll
    for (int u = 0; u < U; ++u) acc += (real && 64 * u + lane < n4 ? wk : 0.f) * (x[g][u] * v[g][u]);
  }
  const float s = wave_sum((acc.x + acc.y) + (acc.z + acc.w));
  if (lane == 0) y[(long long)t * m.d + j] = s + same * h[(long long)t * m.d + j];
}

// ---- many tokens -------------------------------------------------------------------------------
// A wavefront chooses for one token after the other; the places of a workgroup's tokens among an expert's rows
// are counted in LDS, and one addition per expert to the expert's counter gives where they begin.  tokens: per
// workgroup.
__global__ __launch_bounds__(256) void moe_select_kernel(MoeShape m, const float *__restrict__ correction,
                                                         const float *__restrict__ logits, int stride, int T, int tokens,
                                                         int *__restrict__ ids, float *__restrict__ weights,
                                                         int *__restrict__ rank, int *counts) {
  extern __shared__ float smem[];  // per wavefront: s, c, best, weights, ids; then [experts] counts
  const int n = m.experts + m.identity, wave = threadIdx.x >> 6, per_wave = 2 * n + m.groups + 2 * m.top;
  float *s = smem + wave * per_wave, *wl = s + 2 * n + m.groups;
  int *il = (int *)(wl + m.top), *cnt = (int *)(smem + 4 * per_wave);
  for (int e = threadIdx.x; e < m.experts; e += 256) cnt[e] = 0;
  __syncthreads();
  const int t0 = blockIdx.x * tokens;
  for (int i = wave; i < tokens && t0 + i < T; i += 4) {
    const int t = t0 + i;
    choose(m, logits + (long long)t * stride, correction, s, s + n, s + 2 * n, il, wl);
    for (int k = threadIdx.x & 63; k < m.top; k += 64) {
      const int e = il[k];
      ids[t * m.top + k] = e;
      weights[t * m.top + k] = wl[k];
      rank[t * m.top + k] = e < m.experts ? atomicAdd(cnt + e, 1) : 0;
    }
    __threadfence_block();
  }
  __syncthreads();
  for (int e = threadIdx.x; e < m.experts; e += 256) cnt[e] = cnt[e] ? atomicAdd(counts + e, cnt[e]) : 0;
  __syncthreads();
  const int mine = min(tokens, T - t0) * m.top;
  for (int i = threadIdx.x; i < mine; i += 256) {  // (ids and ranks of this workgroup's own tokens)
    const int at = t0 * m.top + i, e = ids[at];
    if (e < m.experts) rank[at] += cnt[e];
  }
}

// Where the experts' rows and tiles begin, which every workgroup works out for itself (the first leaves it), and the rows' tokens in
// the experts' order.  Bound by a launch and two round trips.  In two launches, one workgroup of them with ten steps of a scan through
// LDS, 3.9 + 0.8 + 2.9 us (777 tokens of six); this 4.7
__global__ __launch_bounds__(1024) void moe_rows_kernel(int n, int top, int experts, int tile, const int *__restrict__ counts,
                                                        const int *__restrict__ ids, const int *__restrict__ rank, int *__restrict__ off,
                                                        int *__restrict__ tile_off, int *__restrict__ rows) {
  __shared__ int begins[1024], waves[2][16];
  const int e = threadIdx.x, lane = e & 63, wave = e >> 6, i = blockIdx.x * 1024 + e, at = min(i, n - 1);
  const int mine = ids[at], place = rank[at];
  const int c = counts[min(e, experts - 1)], own = e < experts ? c : 0, tiles = (own + tile - 1) / tile;
  int a = own, b = tiles;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int x = __shfl_up(a, o), y = __shfl_up(b, o);
    a += lane >= o ? x : 0;
    b += lane >= o ? y : 0;
  }
  if (lane == 63) waves[0][wave] = a, waves[1][wave] = b;
  __syncthreads();
  for (int w = 0; w < wave; ++w) {
    a += waves[0][w];
    b += waves[1][w];
  }
  begins[e] = a - own;
  if (blockIdx.x == 0 && e < experts) {
    off[e + 1] = a;
    tile_off[e + 1] = b;
    if (e == 0) off[0] = tile_off[0] = 0;
  }
  __syncthreads();
  if (i < n && mine < experts) rows[begins[mine] + place] = i / top;
}

// Rows of x (gathered, or as they lie) times the matrices of their groups, [N, K] (SWIGLU: [2N, K], gate
// rows and up rows): a product whose operands both run along K, on the bf16 matrix cores with every operand as
// the exact sum of three bf16 numbers (split_mfma.hpp).  A workgroup of four wavefronts, two by two, takes 64 MB
// rows and 128 matrix rows, a wavefront MB x 2 blocks of 32 x 32.  Per step of 16 along K both tiles go
// global memory -> registers (two steps ahead) -> split -> LDS (two stages), where 16-byte units [part][octet of
// k][row] are the fragments of an MFMA.  With SWIGLU a wavefront's first block of matrix rows is gates and the second
// their partners, so that a lane holds both halves of its outputs.
// 777 tokens, 145 rows an expert, 1024 -> 512 gate | up with SwiGLU 157 -> 86 us, 512 -> 1024 84 -> 48 us against the
// fp32 instruction in tiles of 64 rows.  PARTS 1: the matrices' values are bf16 numbers, the products with their other two
// parts, zeros, are left out, and a step is 32 along K, whole 128-byte lines of a row: 85 -> 51 and 49 -> 34 us (150
// tokens 61 -> 31 and 34 -> 17), of which loads that hang on no condition are 14 and 5.
struct GroupedArgs {
  const float *x;
  const int *gather;       // row r of the product is row gather[r] of x; null: row r
  const int *off, *tile_off;  // [groups + 1]; null: one group of `rows` rows
  const float *w;
  float *y;                // [rows, N]
  int rows, groups, K, N;
  bool w_bf16;             // every value of w is a bf16 number (PARTS = 1: the other two parts, zeros, are left out)
};
// LOADS: how pieces of four k are read.  kScalar: any K; kPieces: K a multiple of 4; kSteps: of a step, and no more to it.
enum { kScalar, kPieces, kSteps };
template <int MB, bool SWIGLU, int LOADS, int PARTS>
__global__ __launch_bounds__(256, 2) void moe_product_kernel(const GroupedArgs g) {
  constexpr int HK = PARTS == 1 ? 2 : 1, TK = 16 * HK, TM = 64 * MB, TN = 128;
  constexpr int PER = 4 * HK, kRows = 256 / PER;       // threads that share a row's step, rows that all threads read at once
  constexpr int NA = TM / kRows, NW = TN / kRows;      // 16-byte pieces per thread and step
  constexpr int kPad = HK == 2 ? 2 : 4;                // (the octets of a row in different banks)
  constexpr int kOctX = TM + kPad, kOctW = TN + kPad, kPartX = 2 * HK * kOctX, kPartW = 2 * HK * kOctW;  // units of 16 bytes
  __shared__ __attribute__((aligned(16))) u32x4 lds[2][3 * kPartX + PARTS * kPartW];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int columns = (g.N + (SWIGLU ? TN / 2 : TN) - 1) / (SWIGLU ? TN / 2 : TN);
  int grp = 0, tm = blockIdx.x / columns, r0 = 0, r1 = g.rows;
  if (g.tile_off) {
    if (tm >= g.tile_off[g.groups]) return;
    for (int e0 = 0; e0 < g.groups; e0 += 64)
      grp += (int)__popcll(__ballot(e0 + lane < g.groups && tm >= g.tile_off[min(e0 + lane, g.groups - 1) + 1]));
    grp = __builtin_amdgcn_readfirstlane(grp);
    tm -= g.tile_off[grp];
    r0 = g.off[grp];
    r1 = g.off[grp + 1];
  }
  const int m0 = r0 + tm * TM;
  if (m0 >= r1) return;
  const int K = g.K, N = g.N, o0 = blockIdx.x % columns * (SWIGLU ? TN / 2 : TN);
  const float *w = g.w + (long long)grp * (SWIGLU ? 2 : 1) * N * K;
  // the matrix row behind row i of the tile
  auto matrix_row = [&](int i) {
    return SWIGLU ? (i >> 5 & 1) * N + min(o0 + (i >> 6) * 32 + (i & 31), N - 1) : min(o0 + i, N - 1);
  };

  // piece u of a thread: four k, tid % PER, of tile row tid / PER + kRows u
  const int srow = threadIdx.x / PER, k4 = 4 * (threadIdx.x % PER);
  const float *ap[NA], *bp[NW];
#pragma unroll
  for (int u = 0; u < NA; ++u) {
    const int r = min(m0 + srow + kRows * u, r1 - 1);
    ap[u] = g.x + (long long)(g.gather ? g.gather[r] : r) * K;
  }
#pragma unroll
  for (int u = 0; u < NW; ++u) bp[u] = w + (long long)matrix_row(srow + kRows * u) * K;
  unsigned a_off[NA], b_off[NW];  // kSteps: bytes from a step's first column of row 0 (under 4 GiB: checked at launch)
#pragma unroll
  for (int u = 0; u < NA; ++u) a_off[u] = (unsigned)((ap[u] - g.x + k4) * 4);
#pragma unroll
  for (int u = 0; u < NW; ++u) b_off[u] = (unsigned)((bp[u] - w + k4) * 4);
  f32x4 sa[2][NA], sb[2][NW];
  auto piece = [&](const float *p, int k) {
    if constexpr (LOADS == kScalar) return f32x4{p[min(k, K - 1)], p[min(k + 1, K - 1)], p[min(k + 2, K - 1)], p[min(k + 3, K - 1)]};
    return *(const f32x4 *)(p + min(k, K - 4));
  };
  // what lies behind the end of K counts as zeros
  auto inside = [&](f32x4 v, int k) {
    if constexpr (LOADS == kScalar) return f32x4{k < K ? v.x : 0.f, k + 1 < K ? v.y : 0.f, k + 2 < K ? v.z : 0.f, k + 3 < K ? v.w : 0.f};
    return LOADS == kPieces && k >= K ? f32x4{0.f, 0.f, 0.f, 0.f} : v;
  };
  // (steps behind the last one repeat it, which nobody reads.  No load hangs on a condition: the branches around them had
  // the loop wait for every load it had just issued: 75 rows of 1023 -> 511 by weights of three parts 92 -> 75 us)
  const int last = (K - 1) / TK * TK;
  // Rows of K floats lie a power of two apart, most often, and tiles that all begin at their first column ask the same few memory
  // channels for all of their rows at once: they begin apart (by column tile alone: the order of a row's sums does not depend on other
  // rows).  75 rows of 1024 -> 2 x 512 29.4 -> 25.5 us, 777 rows 50.9 -> 49.6; tiles of 128 rows, which read W half as often, are level
  // or slower.
  const int start = MB == 1 && LOADS == kSteps ? (int)((unsigned)(blockIdx.x % columns) * 5u % (unsigned)(K / TK)) * TK : 0;
  auto load = [&](int set, int k0) {
    k0 = min(k0, last);
    if constexpr (MB == 1 && LOADS == kSteps) k0 = k0 + start > last ? k0 + start - K : k0 + start;
    const int k = k0 + k4;
#pragma unroll
    for (int u = 0; u < NA; ++u)
      sa[set][u] = LOADS == kSteps ? load_at((const f32x4 *)(g.x + k0), a_off[u]) : piece(ap[u], k);
#pragma unroll
    for (int u = 0; u < NW; ++u)
      sb[set][u] = LOADS == kSteps ? load_at((const f32x4 *)(w + k0), b_off[u]) : piece(bp[u], k);
  };
  auto park = [&](int set, int k0, u32x4 *stage) {  // k0: the step's
    u32x2 *at = (u32x2 *)(stage + (k4 >> 3) * kOctX + srow) + (k4 >> 2 & 1);
#pragma unroll
    for (int u = 0; u < NA; ++u)
      split_quad(inside(sa[set][u], k0 + k4) * kLift, at[2 * kRows * u], at[2 * (kRows * u + kPartX)], at[2 * (kRows * u + 2 * kPartX)]);
    at = (u32x2 *)(stage + 3 * kPartX + (k4 >> 3) * kOctW + srow) + (k4 >> 2 & 1);
#pragma unroll
    for (int u = 0; u < NW; ++u) {
      const f32x4 v = inside(sb[set][u], k0 + k4) * kLift;
      if constexpr (PARTS == 3)
        split_quad(v, at[2 * kRows * u], at[2 * (kRows * u + kPartW)], at[2 * (kRows * u + 2 * kPartW)]);
      else
        at[2 * kRows * u] = u32x2{pack_high(v.x, v.y), pack_high(v.z, v.w)};
    }
  };
  const int n = lane & 31, half = lane >> 5, rw = wave & 1, cw = wave >> 1;
  const int a_unit = half * kOctX + rw * 32 * MB + n, b_unit = 3 * kPartX + half * kOctW + cw * 64 + n;
  f32x16 acc[MB][2];
#pragma unroll
  for (int a = 0; a < MB; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;

  const int steps = (K + TK - 1) / TK;
  load(0, 0);
  load(1, TK);
  __builtin_amdgcn_sched_barrier(0);  // (the loop waits for its loads in the order they have here)
  park(0, 0, lds[0]);
  load(0, 2 * TK);
  __syncthreads();
  auto step = [&](int kt, int set) {  // set: holds step kt + 1
    const u32x4 *stage = lds[kt & 1];
    u32x4 af[HK][3][MB], bf[HK][PARTS][2];
#pragma unroll
    for (int h = 0; h < HK; ++h)
#pragma unroll
      for (int p = 0; p < 3; ++p) {
#pragma unroll
        for (int a = 0; a < MB; ++a) af[h][p][a] = stage[a_unit + p * kPartX + 2 * h * kOctX + 32 * a];
#pragma unroll
        for (int b = 0; b < 2 && p < PARTS; ++b) bf[h][p][b] = stage[b_unit + p * kPartW + 2 * h * kOctW + 32 * b];
      }
    park(set, min((kt + 1) * TK, last), lds[(kt & 1) ^ 1]);
    load(set, (kt + 3) * TK);
#pragma unroll
    for (int h = 0; h < HK; ++h)
#pragma unroll
      for (int p = 0; p < 6; ++p) {
        if (kPartB[p] >= PARTS) continue;
#pragma unroll
        for (int a = 0; a < MB; ++a)
#pragma unroll
          for (int b = 0; b < 2; ++b) acc[a][b] = mfma_bf16(af[h][kPartA[p]][a], bf[h][kPartB[p] < PARTS ? kPartB[p] : 0][b], acc[a][b]);
      }
    if constexpr (PARTS == 1 && LOADS == kSteps) {
      // fragments, and then splits, stores and loads handed out between the MFMAs, the loads behind the half of them (masks: 0x100
      // reads of LDS, 2 vector instructions, 8 MFMAs, 0x200 stores to LDS, 0x20 loads).  777 rows of 2048 -> 2 x 768 165 -> 149 us, 768 ->
      // 2048 103 -> 92; of 1024 -> 2 x 512 51.8 -> 50.9; the loads left where they fell: 158 and 97
      __builtin_amdgcn_sched_group_barrier(0x100, HK * (3 * MB + 2), 0);
      __builtin_amdgcn_sched_group_barrier(0x2, 16, 0);
#pragma unroll
      for (int i = 0; i < 12 * MB; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x2, 8, 0);
        __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
        if (i >= 6) __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);
      }
    }
    __syncthreads();
  };
  for (int kt = 1; kt < steps; kt += 2) {  // (in pairs: a way out between them costs waits, too)
    step(kt - 1, 1);
    step(kt, 0);
  }
  if (steps & 1) step(steps - 1, 1);

  // sums that are not finite come from operands that are not (or overflow): again in fp32, which says which (777
  // tokens of width 2048, the fifth NaN: 2.8 ms a layer with its copies against 1.6 without; one k at a time it was 73)
  const int row0 = m0 + rw * 32 * MB + 4 * half;
  float probe = 0.f;
#pragma unroll
  for (int a = 0; a < MB; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) probe = fmaf(acc[a][b][r], 0.f, probe);
  if (__any(probe != 0.f)) {
    const float *xr[MB], *wr[2];
#pragma unroll
    for (int a = 0; a < MB; ++a) {
      const int row = min(m0 + (rw * MB + a) * 32 + n, r1 - 1);
      xr[a] = g.x + (long long)(g.gather ? g.gather[row] : row) * K;
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;
    }
#pragma unroll
    for (int b = 0; b < 2; ++b) wr[b] = w + (long long)matrix_row(cw * 64 + 32 * b + n) * K;
#pragma clang loop unroll(disable)
    for (int k0 = 0; k0 < K; k0 += 8) {  // four of eight k a lane half's
      f32x4 xv[MB], wv[2];
      const int k = k0 + 4 * half;
#pragma unroll
      for (int a = 0; a < MB; ++a) xv[a] = inside(piece(xr[a], k), k);
#pragma unroll
      for (int b = 0; b < 2; ++b) wv[b] = inside(piece(wr[b], k), k);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int a = 0; a < MB; ++a)
#pragma unroll
          for (int b = 0; b < 2; ++b) acc[a][b] = mfma_f32(xv[a][i], wv[b][i], acc[a][b]);
    }
  } else {
#pragma unroll
    for (int a = 0; a < MB; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) acc[a][b] *= kDrop;
  }
#pragma unroll
  for (int a = 0; a < MB; ++a)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = row0 + 32 * a + 8 * (r >> 2) + (r & 3);
      if (row >= r1) continue;
      float *yr = g.y + (long long)row * N;
      if constexpr (SWIGLU) {
        const int col = o0 + cw * 32 + n;
        if (col < N) yr[col] = swiglu1(acc[a][0][r], acc[a][1][r]);
      } else {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const int col = o0 + cw * 64 + 32 * b + n;
          if (col < N) yr[col] = acc[a][b][r];
        }
      }
    }
}

// (where a call ends early)
__global__ __launch_bounds__(256) void moe_clear_kernel(int experts, int *counts) {
  for (int e = threadIdx.x; e < experts; e += 256) counts[e] = 0;
}

// y[t] (+)= sum over the slots of weight * the expert's row, in the slots' order.  The first workgroup clears the
// counters for the next call.
template <int W>
__global__ __launch_bounds__(256) void moe_combine_kernel(MoeShape m, const float *__restrict__ h,
                                                          const float *__restrict__ rows_y, const int *__restrict__ ids,
                                                          const float *__restrict__ weights, const int *__restrict__ rank,
                                                          const int *__restrict__ off, int add, float *__restrict__ y,
                                                          int *__restrict__ counts) {
  typedef float vec_t __attribute__((ext_vector_type(W)));
  const int t = blockIdx.x, n = m.d / W;
  if (t == 0 && blockIdx.y == 0)
    for (int e = threadIdx.x; e < m.experts; e += 256) counts[e] = 0;
  for (int i = blockIdx.y * 256 + threadIdx.x; i < n; i += gridDim.y * 256) {
    vec_t s = add ? ((const vec_t *)(y + (long long)t * m.d))[i] : (vec_t)(0.f);
    for (int k = 0; k < m.top; ++k) {
      const int e = ids[t * m.top + k];
      const float *src = e < m.experts ? rows_y + (long long)(off[e] + rank[t * m.top + k]) * m.d : h + (long long)t * m.d;
      s += weights[t * m.top + k] * ((const vec_t *)src)[i];
    }
    ((vec_t *)(y + (long long)t * m.d))[i] = s;
  }
}

// floats to the next multiple of 16 bytes' worth
size_t up4(size_t n) { return (n + 3) / 4 * 4; }

struct ManyLayout {
  size_t weights, ids, rank, off, tile_off, rows, hidden, rows_y, total;
};
ManyLayout many_layout(const MoeShape &m, int T) {
  ManyLayout l;
  const size_t slots = (size_t)T * m.top;
  size_t at = 0;
  auto take = [&](size_t k) {
    const size_t here = at;
    at += up4(k);
    return here;
  };
  l.weights = take(slots);
  l.ids = take(slots);
  l.rank = take(slots);
  l.off = take((size_t)m.experts + 1);
  l.tile_off = take((size_t)m.experts + 1);
  l.rows = take(slots);
  l.hidden = take(slots * m.ff);
  l.rows_y = take(slots * m.d);
  l.total = at;
  return l;
}

template <int MB, int PARTS>
hipError_t launch_product_tm(const GroupedArgs &g, bool swiglu, hipStream_t stream) {
  constexpr int TM = 64 * MB, TN = 128;
  const long long tiles = g.tile_off ? (long long)g.rows / TM + (g.groups < g.rows ? g.groups : g.rows) : ((long long)g.rows + TM - 1) / TM;
  const int cols = swiglu ? TN / 2 : TN, ny = (g.N + cols - 1) / cols;
  // (columns fastest: with eight blocks of columns the tiles of an expert's rows meet its matrix in one XCD's L2)
  if (tiles < 1 || tiles * ny > 0x7fffffff) return hipErrorInvalidValue;
  const dim3 grid((unsigned)(tiles * ny));
  const bool vec = (g.K & 3) == 0 && !(((uintptr_t)g.x | (uintptr_t)g.w) & 15);
  const int loads = !vec ? kScalar : g.K % (PARTS == 1 ? 32 : 16) || (long long)(g.rows > 2 * g.N ? g.rows : 2 * g.N) * g.K >= 1LL << 30 ? kPieces : kSteps;
#define SHAINET_MOE_PRODUCT(SWIGLU_, LOADS_) \
  hipLaunchKernelGGL((moe_product_kernel<MB, SWIGLU_, LOADS_, PARTS>), grid, dim3(256), 0, stream, g)
  if (swiglu && loads == kSteps)
    SHAINET_MOE_PRODUCT(true, kSteps);
  else if (swiglu && loads == kPieces)
    SHAINET_MOE_PRODUCT(true, kPieces);
  else if (swiglu)
    SHAINET_MOE_PRODUCT(true, kScalar);
  else if (loads == kSteps)
    SHAINET_MOE_PRODUCT(false, kSteps);
  else if (loads == kPieces)
    SHAINET_MOE_PRODUCT(false, kPieces);
  else
    SHAINET_MOE_PRODUCT(false, kScalar);
#undef SHAINET_MOE_PRODUCT
  return hipGetLastError();
}

hipError_t launch_product(const GroupedArgs &g, int tm, bool swiglu, hipStream_t stream) {
  if (g.w_bf16) return tm == 128 ? launch_product_tm<2, 1>(g, swiglu, stream) : launch_product_tm<1, 1>(g, swiglu, stream);
  return tm == 128 ? launch_product_tm<2, 3>(g, swiglu, stream) : launch_product_tm<1, 3>(g, swiglu, stream);
}

}  // namespace

bool moe_shape_ok(const MoeShape &m) {
  const int n = m.experts + m.identity;
  return m.d > 0 && m.ff > 0 && m.experts > 0 && m.identity >= 0 && n <= kMaxRouterOutputs && m.groups > 0 && n % m.groups == 0 &&
         m.keep > 0 && m.keep <= m.groups && m.top > 0 && m.top <= m.keep * (n / m.groups) && m.shared_ff >= 0;
}

size_t moe_few_floats(const MoeShape &m, int T) {
  const size_t width = up4(m.ff > m.shared_ff ? m.ff : m.shared_ff);
  return up4((size_t)T * (m.experts + m.identity)) + 2 * up4((size_t)T * m.top) + (size_t)T * (m.top + 1) * width;
}

hipError_t launch_moe_few(const MoeShape &m, const MoeTensors &w, const float *h, float *y, int T, float *scratch,
                          hipStream_t stream, const ResidualArgs *join) {
  if (!moe_shape_ok(m) || T < 1 || T > kMoeFewTokens || !h || !y || !scratch || !w.router || !w.correction || !w.gate_up ||
      !w.down || (m.shared_ff && (!w.shared_gate_up || !w.shared_down)))
    return hipErrorInvalidValue;
  const int n = m.experts + m.identity, most = m.ff > m.shared_ff ? m.ff : m.shared_ff, width = (int)up4(most);
  float *logits = scratch, *weights = logits + up4((size_t)T * n);
  int *ids = (int *)(weights + up4((size_t)T * m.top));
  float *hidden = (float *)ids + up4((size_t)T * m.top);
  const int shared_blocks = (m.shared_ff + 3) / 4, slot_blocks = (m.ff + 3) / 4;
  const long long blocks = (long long)shared_blocks + (long long)m.top * slot_blocks;
  const dim3 g1((unsigned)((n + 3) / 4), (unsigned)T), g2((unsigned)blocks, (unsigned)T), g3((unsigned)((m.d + 3) / 4), (unsigned)T);
  const size_t lds = ((size_t)up4(m.d) + 2 * n + m.groups + 2 * m.top) * sizeof(float);
  if (blocks > 0x7fffffffLL || lds > 64 * 1024) return hipErrorInvalidValue;
  const bool vec_d = (m.d & 3) == 0, vec_ff = ((m.ff | m.shared_ff) & 3) == 0;
  if (join && (T != 1 || join->h != h || join->d != m.d)) return hipErrorInvalidValue;
  const bool joins = join && row_join_fits(*join) && !((uintptr_t)w.router & 15);
  if (join && !joins) {
    const hipError_t e = launch_residual(*join, stream);
    if (e != hipSuccess) return e;
  }
  if (vec_d) {
    if (joins && m.d == 1024)
      hipLaunchKernelGGL(moe_join_logits_kernel<1>, g1, dim3(256), 0, stream, *join, w.router, logits, n);
    else if (joins)
      hipLaunchKernelGGL(moe_join_logits_kernel<2>, g1, dim3(256), 0, stream, *join, w.router, logits, n);
    else
      hipLaunchKernelGGL(moe_logits_kernel<true>, g1, dim3(256), 0, stream, h, w.router, logits, n, m.d);
    hipLaunchKernelGGL(moe_up_kernel<true>, g2, dim3(256), lds, stream, m, w, h, logits, hidden, width, shared_blocks, slot_blocks,
                       ids, weights);
  } else {
    hipLaunchKernelGGL(moe_logits_kernel<false>, g1, dim3(256), 0, stream, h, w.router, logits, n, m.d);
    hipLaunchKernelGGL(moe_up_kernel<false>, g2, dim3(256), lds, stream, m, w, h, logits, hidden, width, shared_blocks, slot_blocks,
                       ids, weights);
  }
  const int spans = (m.ff + 255) / 256;
#define SHAINET_MOE_DOWN(U_, G_) \
  hipLaunchKernelGGL((moe_down_once_kernel<U_, G_>), g3, dim3(256), 0, stream, m, w, h, hidden, width, ids, weights, y)
#define SHAINET_MOE_DOWN_SLOTS(U_) \
  do {                             \
    if (m.top <= 2)                \
      SHAINET_MOE_DOWN(U_, 2);     \
    else if (m.top <= 4)           \
      SHAINET_MOE_DOWN(U_, 4);     \
    else                           \
      SHAINET_MOE_DOWN(U_, 8);     \
  } while (0)
  if (vec_ff && m.top <= 8 && spans == 1)
    SHAINET_MOE_DOWN_SLOTS(1);
  else if (vec_ff && m.top <= 8 && spans == 2)
    SHAINET_MOE_DOWN_SLOTS(2);
  else if (vec_ff && m.top <= 8 && spans == 3)
    SHAINET_MOE_DOWN_SLOTS(3);
  else if (vec_ff)
    hipLaunchKernelGGL(moe_down_kernel<true>, g3, dim3(256), 0, stream, m, w, h, hidden, width, ids, weights, y);
  else
    hipLaunchKernelGGL(moe_down_kernel<false>, g3, dim3(256), 0, stream, m, w, h, hidden, width, ids, weights, y);
#undef SHAINET_MOE_DOWN_SLOTS
#undef SHAINET_MOE_DOWN
  return hipGetLastError();
}

size_t moe_many_floats(const MoeShape &m, int T) { return many_layout(m, T).total; }

hipError_t launch_moe_many(const MoeShape &m, const MoeTensors &w, const float *h, const float *logits, int stride, float *y,
                           bool add_to_y, int T, float *scratch, int *counts, hipStream_t stream) {
  if (!moe_shape_ok(m) || T < 1 || (long long)T * m.top > 0x3fffffff || !h || !y || !logits ||
      stride < m.experts + m.identity || !scratch || !counts || !w.correction || !w.gate_up || !w.down)
    return hipErrorInvalidValue;
  const ManyLayout l = many_layout(m, T);
  const int n = m.experts + m.identity, slots = T * m.top;
  float *weights = scratch + l.weights, *hidden = scratch + l.hidden, *rows_y = scratch + l.rows_y;
  int *ids = (int *)(scratch + l.ids), *rank = (int *)(scratch + l.rank), *off = (int *)(scratch + l.off),
      *tile_off = (int *)(scratch + l.tile_off), *rows = (int *)(scratch + l.rows);
  hipError_t e = hipSuccess;
  const size_t lds = ((size_t)4 * (2 * n + m.groups + 2 * m.top) + m.experts) * sizeof(float);
  if (lds > 64 * 1024) return hipErrorInvalidValue;
  const int tokens = T <= 4096 ? 4 : 16;
  hipLaunchKernelGGL(moe_select_kernel, dim3((unsigned)((T + tokens - 1) / tokens)), dim3(256), lds, stream, m, w.correction, logits,
                     stride, T, tokens, ids, weights, rank, counts);
  // per_expert: rows an expert gets if the router spreads them evenly.  Tiles of 128 rows split each matrix half as often
  // and fill up worse.  Prompts, 64 | 128, us, rows an expert by width and expert width:
  //               25           75           125          194          260          375
  //   1024,  512  949 | 977    1145 | 1194  1264 | 1268  1474 | 1405  1627 | 1654  2060 | 2052   (281: 1890 | 2060)
  //   1024, 1024  1092 | 1109  1343 | 1331  1504 | 1608  1864 | 1750  2098 | 2037  2706 | 2550
  //   1536,  768  1158 | 1235  1466 | 1446  1635 | 1533  2163 | 2174  2523 | 2434  3063 | 2963
  //   2048,  512  1257 | 1298  1473 | 1510  1714 | 1760  2260 | 2089  2730 | 2721  3647 | 3295
  //   2048,  768  1460 | 1489  1866 | 1827  2278 | 2244  3280 | 3177  4045 | 3926  5520 | 5363
  //   2048, 1024  1469 | 1451  1895 | 1763  2272 | 2486  3127 | 2866  3766 | 3395  4910 | 4292
  //   4096,  512  1845 | 2000  2351 | 2472  2817 | 2842  3946 | 3697  5138 | 4781  6469 | 5960
  // (2048, 768: the last at 425).  Tiles of 32 lose 4 to 23 % everywhere, one row included.
  const int per_expert = slots / n, best_tm = per_expert > ((long long)m.d * m.ff > 512 << 10 ? 160 : 320) ? 128 : 64;
  // a tuning knob: 64 or 128 (32, which there once was, is 64)
  static const int tile_knob = getenv("SHAINET_HIP_MOE_TILE") ? atoi(getenv("SHAINET_HIP_MOE_TILE")) : 0;
  const int tm = tile_knob == 128 ? 128 : tile_knob == 64 || tile_knob == 32 ? 64 : best_tm;
  hipLaunchKernelGGL(moe_rows_kernel, dim3((unsigned)((slots + 1023) / 1024)), dim3(1024), 0, stream, slots, m.top, m.experts, tm,
                     counts, ids, rank, off, tile_off, rows);
  GroupedArgs g = {};
  g.x = h;
  g.gather = rows;
  g.off = off;
  g.tile_off = tile_off;
  g.w = w.gate_up;
  g.w_bf16 = w.gate_up_bf16;
  g.y = hidden;
  g.rows = slots;
  g.groups = m.experts;
  g.K = m.d;
  g.N = m.ff;
  auto ended = [&]() {
    hipLaunchKernelGGL(moe_clear_kernel, dim3(1), dim3(256), 0, stream, m.experts, counts);
    return e;
  };
  if ((e = launch_product(g, tm, true, stream)) != hipSuccess) return ended();
  g.x = hidden;
  g.gather = nullptr;
  g.w = w.down;
  g.w_bf16 = w.down_bf16;
  g.y = rows_y;
  g.K = m.ff;
  g.N = m.d;
  if ((e = launch_product(g, tm, false, stream)) != hipSuccess) return ended();
  const bool vec = (m.d & 3) == 0;
  const int per = vec ? 1024 : 256;
  const dim3 grid((unsigned)T, (unsigned)((m.d + per - 1) / per));
  if (vec)
    hipLaunchKernelGGL(moe_combine_kernel<4>, grid, dim3(256), 0, stream, m, h, rows_y, ids, weights, rank, off, add_to_y ? 1 : 0, y, counts);
  else
    hipLaunchKernelGGL(moe_combine_kernel<1>, grid, dim3(256), 0, stream, m, h, rows_y, ids, weights, rank, off, add_to_y ? 1 : 0, y, counts);
  e = hipGetLastError();
  return e == hipSuccess ? e : ended();
}

}  // namespace shainet
