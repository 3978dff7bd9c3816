// The kernels of a LlamaBlock around attention, and of the steps after the last
// block, for gfx950.  They restate the reference's host loops with its number
// types, so that results agree with its CPU path to the last bit or two:
//   RMSNorm#forward        rms_norm.cr:18-37   sum of squares, the root and the
//                                              scaling in fp64, one rounding to fp32
//   SimpleMatrix#+         simple_matrix.cr:39-48   fp64 add, rounded to fp32
//   SwiGLUFF#forward       swiglu_ff.cr:76-91  g / (1 + exp(-g)) * up in fp64
//   EmbeddingLayer#embed_cpu   embedding_layer.cr:129-153   row gather
//   Sampler                text/sampler.cr:38-120   greedy, repetition penalty, top-k
// All of them are bound by HBM (or by latency at decode sizes); fp64 arithmetic is
// free at these intensities on this part.
#include "activation.hpp"
#include "block_kernels.hpp"
#include "split_mfma.hpp"

#include <math.h>
#include <stdint.h>

namespace shainet {

namespace {

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// One workgroup per row.
__global__ __launch_bounds__(256) void rmsnorm_kernel(const float *__restrict__ x, long long x_stride,
                                                      const float *__restrict__ gamma, float *__restrict__ out,
                                                      int cols, double eps, bool planes) {
  __shared__ double red[4];
  const float *xr = x + (long long)blockIdx.x * x_stride;
  float *orow = out + (long long)blockIdx.x * cols;
  const bool vec = (cols & 3) == 0 && (x_stride & 3) == 0;
  double sq = 0.0;
  if (vec) {
    for (int j = threadIdx.x * 4; j < cols; j += 1024) {
      const f32x4 v = *(const f32x4 *)(xr + j);
      sq += (double)v.x * (double)v.x + (double)v.y * (double)v.y;
      sq += (double)v.z * (double)v.z + (double)v.w * (double)v.w;
    }
  } else {
    for (int j = threadIdx.x; j < cols; j += 256) sq += (double)xr[j] * (double)xr[j];
  }
  sq = wave_sum(sq);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sq;
  __syncthreads();
  const double total = (red[0] + red[1]) + (red[2] + red[3]);
  const double rms = sqrt(total / (double)cols + eps);
  if (vec) {
    for (int j = threadIdx.x * 4; j < cols; j += 1024) {
      const f32x4 v = *(const f32x4 *)(xr + j);
      f32x4 gm = {1.f, 1.f, 1.f, 1.f};
      if (gamma) gm = *(const f32x4 *)(gamma + j);
      f32x4 y;
      y.x = (float)(((double)v.x / rms) * (double)gm.x);
      y.y = (float)(((double)v.y / rms) * (double)gm.y);
      y.z = (float)(((double)v.z / rms) * (double)gm.z);
      y.w = (float)(((double)v.w / rms) * (double)gm.w);
      if (planes)
        store_planes(out, blockIdx.x, gridDim.x, j, cols, y);
      else
        *(f32x4 *)(orow + j) = y;
    }
  } else {
    for (int j = threadIdx.x; j < cols; j += 256)
      orow[j] = (float)(((double)xr[j] / rms) * (double)(gamma ? gamma[j] : 1.f));
  }
}

__global__ __launch_bounds__(256) void add_kernel(const float *__restrict__ a, const float *__restrict__ b,
                                                  float *__restrict__ out, long long n) {
  const long long i = ((long long)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i + 3 < n) {
    const f32x4 x = *(const f32x4 *)(a + i), y = *(const f32x4 *)(b + i);
    f32x4 r;
    r.x = (float)((double)x.x + (double)y.x);
    r.y = (float)((double)x.y + (double)y.y);
    r.z = (float)((double)x.z + (double)y.z);
    r.w = (float)((double)x.w + (double)y.w);
    *(f32x4 *)(out + i) = r;
  } else {
    for (long long j = i; j < n; ++j) out[j] = (float)((double)a[j] + (double)b[j]);
  }
}

__global__ __launch_bounds__(256) void copy_floats_kernel(const float *__restrict__ x, float *__restrict__ out, long long n) {
  const long long i = ((long long)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i + 3 < n && !(((uintptr_t)x | (uintptr_t)out) & 15)) {
    *(f32x4 *)(out + i) = *(const f32x4 *)(x + i);
  } else {
    for (long long j = i; j < n && j < i + 4; ++j) out[j] = x[j];
  }
}

__global__ __launch_bounds__(256) void swiglu_act_kernel(const float *__restrict__ gate_up, float *__restrict__ hidden,
                                                         int ff) {
  const int r = blockIdx.y;
  const float *gr = gate_up + (long long)r * 2 * ff;
  float *hr = hidden + (long long)r * ff;
  const int j = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (j + 3 < ff && (ff & 3) == 0) {
    const f32x4 g = *(const f32x4 *)(gr + j), u = *(const f32x4 *)(gr + ff + j);
    *(f32x4 *)(hr + j) = f32x4{swiglu(g.x, u.x), swiglu(g.y, u.y), swiglu(g.z, u.z), swiglu(g.w, u.w)};
  } else {
    for (int k = j; k < ff && k < j + 4; ++k) hr[k] = swiglu(gr[k], gr[ff + k]);
  }
}

__global__ __launch_bounds__(256) void embed_kernel(const float *__restrict__ table, const int *__restrict__ tokens,
                                                    float *__restrict__ out, int d_model, float scale,
                                                    const float *__restrict__ positions) {
  const float *src = table + (long long)tokens[blockIdx.x] * d_model;
  float *dst = out + (long long)blockIdx.x * d_model;
  const float *pos = positions + (positions ? (long long)blockIdx.x * d_model : 0);
  for (int j = threadIdx.x; j < d_model; j += 256) dst[j] = positions ? src[j] * scale + pos[j] : src[j] * scale;
}

// the same for ids that travel in the kernel's arguments
__global__ __launch_bounds__(256) void embed_list_kernel(const float *__restrict__ table, const IdList list,
                                                         float *__restrict__ out, int d_model, float scale,
                                                         const float *__restrict__ positions) {
  const float *src = table + (long long)list.id[blockIdx.x] * d_model;
  float *dst = out + (long long)blockIdx.x * d_model;
  const float *pos = positions + (positions ? (long long)blockIdx.x * d_model : 0);
  for (int j = threadIdx.x; j < d_model; j += 256) dst[j] = positions ? src[j] * scale + pos[j] : src[j] * scale;
}

// Dynamic Tanh: no statistics over the row, so a workgroup takes 1024 columns of one row.
__global__ __launch_bounds__(256) void dyn_tanh_kernel(const float *__restrict__ x, long long x_stride,
                                                       const float *__restrict__ gamma, const float *__restrict__ beta,
                                                       float alpha, float *__restrict__ out, int cols, bool planes) {
  const float *xr = x + (long long)blockIdx.x * x_stride;
  float *orow = out + (long long)blockIdx.x * cols;
  const int j = (blockIdx.y * 256 + threadIdx.x) * 4;
  if (j + 3 < cols && ((cols | x_stride) & 3) == 0) {
    const f32x4 v = *(const f32x4 *)(xr + j), g = *(const f32x4 *)(gamma + j), b = *(const f32x4 *)(beta + j);
    const f32x4 y = {tanhf(alpha * v.x) * g.x + b.x, tanhf(alpha * v.y) * g.y + b.y, tanhf(alpha * v.z) * g.z + b.z,
                     tanhf(alpha * v.w) * g.w + b.w};
    if (planes)
      store_planes(out, blockIdx.x, gridDim.x, j, cols, y);
    else
      *(f32x4 *)(orow + j) = y;
  } else {
    for (int k = j; k < cols && k < j + 4; ++k) orow[k] = tanhf(alpha * xr[k]) * gamma[k] + beta[k];
  }
}

__global__ __launch_bounds__(256) void add_bias_row_kernel(float *__restrict__ logits, const float *__restrict__ bias,
                                                           int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  // matrix[i, j] += b[0, j] on SimpleMatrix: fp64 add, rounded (network_run.cr:221-225)
  if (i < n) logits[i] = (float)((double)logits[i] + (double)bias[i]);
}

// The reference walks the ids in order and rewrites the logit once per occurrence, so an id that repeats is
// penalised repeatedly.  Different ids do not meet: the thread of an id's first place does all its occurrences.
// The ids (a few dozen) travel in the kernel's arguments where they fit, without a copy to the device first.
// 64 ids: 4.2 us; one thread that walks them, a memory round trip each, 22 us.
__device__ __forceinline__ void penalise(float *__restrict__ logits, int vocab, const int *ids, int padded, int i, double p) {
  const int id = ids[i];
  if (id < 0 || id >= vocab) return;
  float v = logits[id];  // (asked for before it is known whether the place is the first: it is in flight meanwhile)
  int times = 0;
  bool first = true;
#pragma unroll 4
  for (int j = 0; j < padded; j += 4) {
    const int4 other = *(const int4 *)(ids + j);
    first = first && !((other.x == id && j < i) || (other.y == id && j + 1 < i) || (other.z == id && j + 2 < i) ||
                       (other.w == id && j + 3 < i));
    times += (other.x == id) + (other.y == id) + (other.z == id) + (other.w == id);
  }
  if (!first) return;
  for (; times > 0; --times) v = (float)(v > 0.f ? (double)v / p : (double)v * p);
  logits[id] = v;
}
// (ids: n of them and -1 up to a multiple of 4)
__global__ __launch_bounds__(256) void repetition_penalty_kernel(float *__restrict__ logits, int vocab,
                                                                 const int *__restrict__ ids, int n, double p) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) penalise(logits, vocab, ids, (n + 3) & ~3, i, p);
}
__global__ __launch_bounds__(256) void repetition_penalty_list_kernel(float *__restrict__ logits, int vocab, const IdList list,
                                                                      int n, double p) {
  __shared__ __attribute__((aligned(16))) int ids[kIdList];
  ids[threadIdx.x] = (int)threadIdx.x < n ? list.id[threadIdx.x] : -1;
  __syncthreads();
  if ((int)threadIdx.x < n) penalise(logits, vocab, ids, (n + 3) & ~3, threadIdx.x, p);
}

// ---- top-k ------------------------------------------------------------------
// A candidate is a 64-bit key: the float's bits mapped to an unsigned integer of
// the same order in the high word, ~index in the low word, so that the largest
// key is the largest value and, among equal values, the smallest index.  Key 0
// means "no candidate".
__device__ __forceinline__ unsigned long long make_key(float v, int idx, bool finite_only) {
  if (v != v) return 0ull;
  if (finite_only && (v == INFINITY || v == -INFINITY)) return 0ull;
  unsigned u = __float_as_uint(v);
  u = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
  // -0.0 and +0.0 compare equal in the reference (v > x is false both ways)
  if (v == 0.f) u = 0x80000000u;
  return ((unsigned long long)u << 32) | (unsigned)(~(unsigned)idx);
}
__device__ __forceinline__ float key_value(unsigned long long key, const float *logits) {
  return logits[~(unsigned)(key & 0xffffffffu)];
}

__device__ __forceinline__ unsigned long long wave_max(unsigned long long v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned long long other = __shfl_xor(v, o);
    v = other > v ? other : v;
  }
  return v;
}

constexpr int kTopkChunk = 2048;   // logits per workgroup in the first pass; 8 keys per thread
constexpr int kTopkThreads = 256;  // >= kMaxTopK
constexpr int kTopkHeld = 4;       // candidates that a thread of the merge holds: 1024 of them, 40 of a vocabulary of 51000

struct TopkLds {
  unsigned long long best[kTopkThreads];   // every thread's largest key
  unsigned long long pool[kTopkChunk];     // keys at or above the threshold, in no order
  unsigned long long win[kMaxTopK];        // the k largest, descending
  unsigned long long threshold;
  int pooled;
};

// The k-th largest of the threads' largest keys has at least k keys at or above it, and hardly more when the
// large keys are spread over the threads.  (Keys are unique but for 0, so equal logits do not crowd the pool.)
__device__ __forceinline__ void topk_threshold(TopkLds &s, unsigned long long mine, int k) {
  // (up to 48 of them: the largest keys of four threads each are enough, and a quarter of the comparisons)
  const bool few = k <= 48;
  if (few) {
#pragma unroll
    for (int o = 1; o <= 2; o <<= 1) {
      const unsigned long long other = __shfl_xor(mine, o);
      mine = other > mine ? other : mine;
    }
  }
  if (!few || (threadIdx.x & 3) == 0) s.best[few ? threadIdx.x >> 2 : threadIdx.x] = mine;
  if (threadIdx.x == 0) s.threshold = 0ull, s.pooled = 0;
  __syncthreads();
  int above = 0;
  if (few) {  // (the four threads that hold a key share the comparisons)
    unsigned long long other[kTopkThreads / 16];
#pragma unroll
    for (int u = 0; u < kTopkThreads / 16; ++u) other[u] = s.best[(threadIdx.x & 3) + 4 * u];
#pragma unroll
    for (int u = 0; u < kTopkThreads / 16; ++u) above += other[u] > mine;
    above += __shfl_xor(above, 1);
    above += __shfl_xor(above, 2);
  } else {
#pragma unroll 16
    for (int j = 0; j < kTopkThreads; ++j) above += s.best[j] > mine;
  }
  if (above == k - 1) s.threshold = mine;  // (of several threads only where they hold the same)
  __syncthreads();
}
// (a wavefront asks for the places of all its keys at once)
template <int N>
__device__ __forceinline__ void topk_pool(TopkLds &s, const unsigned long long (&keys)[N]) {
  const unsigned long long least = s.threshold > 1ull ? s.threshold : 1ull, here = __ballot(true);
  const int lane = threadIdx.x & 63;
  int place[N], n = 0;
#pragma unroll
  for (int u = 0; u < N; ++u) {
    const unsigned long long taken = __ballot(keys[u] >= least);
    place[u] = n + __popcll(taken & ((1ull << lane) - 1));
    n += __popcll(taken);
  }
  if (n == 0) return;
  int at = 0;
  if (lane == __ffsll(here) - 1) at = atomicAdd(&s.pooled, n);
  at = __builtin_amdgcn_readfirstlane(at);
#pragma unroll
  for (int u = 0; u < N; ++u)
    if (keys[u] >= least && at + place[u] < kTopkChunk) s.pool[at + place[u]] = keys[u];
}
// win = the k largest of the pool in order (0 behind the last one).  Up to 128 of them: four, or two, threads compare a key.
template <int P>
__device__ __forceinline__ void topk_rank_by(TopkLds &s, int k, int n) {
  const int part = threadIdx.x % P;
  for (int i = threadIdx.x / P; i < n; i += kTopkThreads / P) {
    const unsigned long long key = s.pool[i];
    int above = 0;
#pragma unroll 8
    for (int j = part; j < n; j += P) above += s.pool[j] > key;
#pragma unroll
    for (int o = 1; o < P; o <<= 1) above += __shfl_xor(above, o);
    if (part == 0 && above < k) s.win[above] = key;
  }
}
__device__ __forceinline__ void topk_rank(TopkLds &s, int k) {
  __syncthreads();
  const int n = s.pooled;
  if (n <= kTopkThreads / 4)
    topk_rank_by<4>(s, k, n);
  else if (n <= kTopkThreads / 2)
    topk_rank_by<2>(s, k, n);
  else
    topk_rank_by<1>(s, k, n);
  for (int r = n + (int)threadIdx.x; r < k; r += kTopkThreads) s.win[r] = 0ull;
  __syncthreads();
}

// cand[r * chunks + c]: the r-th largest key of chunk c.  Rounds of "take the largest key" took 32 us for
// k = 40 (two barriers a round); a threshold and ranks 8 us, nearly whatever k is; the merge with the draw behind
// it 34 + 8 us and 8.  Bound by their chains: logits asked for one after the other behind a condition, a place in the pool at a time,
// a thread per key that compares it with all others; all at once, a place per wavefront, and up to four threads a key: 5.4 and 5.7.
__global__ __launch_bounds__(kTopkThreads) void topk_chunk_kernel(const float *__restrict__ logits, int vocab, int k,
                                                                  int finite_only, unsigned long long *__restrict__ cand) {
  __shared__ TopkLds s;
  unsigned long long keys[8], mine = 0ull;
  const int base = blockIdx.x * kTopkChunk;
  float v[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) v[u] = logits[min(base + u * kTopkThreads + (int)threadIdx.x, vocab - 1)];
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const int idx = base + u * kTopkThreads + threadIdx.x;
    keys[u] = idx < vocab ? make_key(v[u], idx, finite_only != 0) : 0ull;
    mine = keys[u] > mine ? keys[u] : mine;
  }
  topk_threshold(s, mine, k);
  topk_pool(s, keys);
  topk_rank(s, k);
  if ((int)threadIdx.x < k) cand[(long long)threadIdx.x * gridDim.x + blockIdx.x] = s.win[threadIdx.x];
}

// One workgroup merges the chunks' candidates: their first ones come first, so the largest keys are spread over
// the threads.  With `pick`, the rest of Sampler#sample follows (text/sampler.cr:118-150): the temperature softmax
// over the survivors and the inverse-CDF pick for the uniform draw r, in fp64, its sums in the reference's order.
__global__ __launch_bounds__(kTopkThreads) void topk_merge_kernel(const float *__restrict__ logits,
                                                                  const unsigned long long *__restrict__ cand, int n_cand, int k,
                                                                  int *__restrict__ out_ids, float *__restrict__ out_vals,
                                                                  int *__restrict__ out_count, int fallback_id,
                                                                  int *__restrict__ pick, double temperature, double r) {
  __shared__ TopkLds s;
  __shared__ double weight[kMaxTopK];
  unsigned long long keys[kTopkHeld], mine = 0ull;
#pragma unroll
  for (int u = 0; u < kTopkHeld; ++u) keys[u] = cand[min(u * kTopkThreads + (int)threadIdx.x, n_cand - 1)];
#pragma unroll
  for (int u = 0; u < kTopkHeld; ++u) {
    if (u * kTopkThreads + (int)threadIdx.x >= n_cand) keys[u] = 0ull;
    mine = keys[u] > mine ? keys[u] : mine;
  }
  for (int i = kTopkHeld * kTopkThreads + threadIdx.x; i < n_cand; i += kTopkThreads) mine = cand[i] > mine ? cand[i] : mine;
  topk_threshold(s, mine, k);
  auto pool = [&]() {
    topk_pool(s, keys);
    for (int i = kTopkHeld * kTopkThreads + threadIdx.x; i < n_cand; i += kTopkThreads) {
      const unsigned long long key[1] = {cand[i]};
      topk_pool(s, key);
    }
  };
  pool();
  __syncthreads();
  if (s.pooled > kTopkChunk) {  // too many for the pool: the threshold is raised to the k-th largest key, a bit at a time
    unsigned long long low = 0ull;
    for (int bit = 63; bit >= 0; --bit) {
      const unsigned long long tried = low | (1ull << bit);
      __syncthreads();
      if (threadIdx.x == 0) s.pooled = 0;
      __syncthreads();
      int here = 0;
      for (int i = threadIdx.x; i < n_cand; i += kTopkThreads) here += cand[i] >= tried;
      atomicAdd(&s.pooled, here);
      __syncthreads();
      if (s.pooled >= k) low = tried;
    }
    __syncthreads();
    if (threadIdx.x == 0) s.threshold = low, s.pooled = 0;
    __syncthreads();
    pool();
  }
  topk_rank(s, k);
  const int n = s.pooled < k ? s.pooled : k, t = threadIdx.x;
  const unsigned long long key = t < k ? s.win[t] : 0ull;
  const float v = key ? key_value(key, logits) : 0.f;
  if (t < k) {
    if (out_ids) out_ids[t] = key ? (int)(~(unsigned)(key & 0xffffffffu)) : fallback_id;
    if (out_vals) out_vals[t] = v;
  }
  if (t == 0 && out_count) *out_count = n;
  if (!pick) return;
  // descending order: element 0 is the maximum
  if (t < n) weight[t] = exp((double)v / temperature - (double)key_value(s.win[0], logits) / temperature);
  __syncthreads();
  if (t != 0) return;
  // (the host may be looking at the word)
  auto say = [&](int id) { __hip_atomic_store(pick, id, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); };
  if (n <= 0) {  // all-NaN row: nothing to sample (sampler.cr:121)
    say(0);
    return;
  }
  double sum = 0.0;
  for (int i = 0; i < n; ++i) sum += weight[i];
  const double inv_sum = 1.0 / sum;
  double cumulative = 0.0;
  int best = n - 1;
  for (int i = 0; i < n; ++i) {
    cumulative += weight[i] * inv_sum;
    if (r <= cumulative) {
      best = i;
      break;
    }
  }
  say((int)(~(unsigned)(s.win[best] & 0xffffffffu)));
}

// Sampler.greedy and the next step's embedding lookup in one launch of one workgroup: *id = the largest finite
// logit's place (0: none), out = its row of the table.  cand null: the logits themselves are read here, 128 KB of
// them (vocabulary of 32000): 4.7 us (6.7 with a 64-bit key for each of them and conditional loads), where two top-k launches and the
// lookup took 11; from 65536 on the chunks' largest keys are (n of them).
__global__ __launch_bounds__(1024) void greedy_embed_kernel(const float *__restrict__ logits, int vocab,
                                                            const unsigned long long *__restrict__ cand, int n,
                                                            int *__restrict__ id, const float *__restrict__ table,
                                                            float *__restrict__ out, int d_model, float scale,
                                                            const float *__restrict__ position) {
  __shared__ unsigned long long red[16];
  unsigned long long best = 0ull;
  if (cand) {
    for (int i = threadIdx.x; i < n; i += 1024) best = cand[i] > best ? cand[i] : best;
  } else {
    const int whole = vocab & ~3;
    float most = -INFINITY;  // (a thread comes by its logits in their order: the first of equals stays)
    int place = 0;
    for (int i0 = 0; i0 < whole; i0 += 8 * 4096) {
      f32x4 v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = *(const f32x4 *)(logits + min(i0 + u * 4096 + 4 * (int)threadIdx.x, whole - 4));
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int i = min(i0 + u * 4096 + 4 * (int)threadIdx.x, whole - 4);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const bool more = v[u][c] > most && v[u][c] < INFINITY;
          most = more ? v[u][c] : most;
          place = more ? i + c : place;
        }
      }
    }
    best = make_key(most, place, true);
    if (whole + (int)threadIdx.x < vocab) {
      const unsigned long long key = make_key(logits[whole + threadIdx.x], whole + threadIdx.x, true);
      best = key > best ? key : best;
    }
  }
  best = wave_max(best);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = best;
  __syncthreads();
  best = red[0];
#pragma unroll
  for (int i = 1; i < 16; ++i) best = red[i] > best ? red[i] : best;
  const int token = best ? (int)(~(unsigned)(best & 0xffffffffu)) : 0;
  if (threadIdx.x == 0) *id = token;
  const float *src = table + (long long)token * d_model;
  for (int j = threadIdx.x; j < d_model; j += 1024) out[j] = position ? src[j] * scale + position[j] : src[j] * scale;
}

// RoPE.apply (rope.cr:7-33): one lane per (row, pair).  Everything in fp64 as the reference has
// it (Float32 operands widened, `theta ** (2.0 * i / head_dim)`, the angle, Math.cos / Math.sin,
// both products and their difference or sum), rounded once when the result is stored.
__global__ __launch_bounds__(256) void rope_apply_kernel(const float *__restrict__ x, float *__restrict__ out,
                                                         int seq_len, int head_dim, int start_pos, double theta) {
  const int half = head_dim / 2;
  const long long per_row = half + (head_dim & 1);  // the odd trailing column rides along as one more item
  const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (long long)seq_len * per_row) return;
  const int pos = (int)(idx / per_row), i = (int)(idx - (long long)pos * per_row);
  const float *xr = x + (long long)pos * head_dim;
  float *orow = out + (long long)pos * head_dim;
  if (i == half) {
    orow[head_dim - 1] = xr[head_dim - 1];
    return;
  }
  const double freq = 1.0 / pow(theta, 2.0 * (double)i / (double)head_dim);
  const double angle = (double)(pos + start_pos) * freq;
  const double c = cos(angle), s = sin(angle);
  const double x0 = (double)xr[i], x1 = (double)xr[i + half];
  orow[i] = (float)(x0 * c - x1 * s);
  orow[i + half] = (float)(x1 * c + x0 * s);
}

// 32 x 32 tiles through LDS: coalesced on both sides
// (row_scale, nullable: row r of src is multiplied by row_scale[r] on its way)
__global__ __launch_bounds__(256) void transpose_kernel(const float *__restrict__ src, float *__restrict__ dst, int rows,
                                                        int cols, const float *__restrict__ row_scale) {
  __shared__ float tile[32][33];
  const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int i = ty; i < 32; i += 8)
    if (r0 + i < rows && c0 + tx < cols)
      tile[i][tx] = src[(long long)(r0 + i) * cols + c0 + tx] * (row_scale ? row_scale[r0 + i] : 1.0f);
  __syncthreads();
  for (int i = ty; i < 32; i += 8)
    if (c0 + i < cols && r0 + tx < rows) dst[(long long)(c0 + i) * rows + r0 + tx] = tile[tx][i];
}

__global__ __launch_bounds__(256) void transposed_differ_kernel(const float *__restrict__ a, const float *__restrict__ b,
                                                                int rows, int cols, int *__restrict__ differ) {
  __shared__ unsigned tile[32][33];
  const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int i = ty; i < 32; i += 8)
    if (r0 + i < rows && c0 + tx < cols) tile[i][tx] = __float_as_uint(a[(long long)(r0 + i) * cols + c0 + tx]);
  __syncthreads();
  bool bad = false;
  for (int i = ty; i < 32; i += 8)
    if (c0 + i < cols && r0 + tx < rows) bad = bad || __float_as_uint(b[(long long)(c0 + i) * rows + r0 + tx]) != tile[tx][i];
  if (bad) *differ = 1;
}

}  // namespace

hipError_t launch_transposed_differ(const float *a, const float *b, int rows, int cols, int *differ, hipStream_t stream) {
  if (!a || !b || !differ || rows < 1 || cols < 1 || (rows + 31) / 32 > 65535) return hipErrorInvalidValue;
  hipLaunchKernelGGL(transposed_differ_kernel, dim3((unsigned)((cols + 31) / 32), (unsigned)((rows + 31) / 32)), dim3(256),
                     0, stream, a, b, rows, cols, differ);
  return hipGetLastError();
}

hipError_t launch_transpose(const float *src, float *dst, int rows, int cols, hipStream_t stream, const float *row_scale) {
  if (!src || !dst || rows < 1 || cols < 1 || (rows + 31) / 32 > 65535) return hipErrorInvalidValue;
  hipLaunchKernelGGL(transpose_kernel, dim3((unsigned)((cols + 31) / 32), (unsigned)((rows + 31) / 32)), dim3(256), 0,
                     stream, src, dst, rows, cols, row_scale);
  return hipGetLastError();
}

hipError_t launch_rmsnorm(const float *x, long long x_stride, const float *gamma, float *out, int rows, int cols,
                          double eps, hipStream_t stream, bool planes) {
  if (rows < 1 || cols < 1 || x_stride < cols || (planes && (cols % 32 || x_stride % 4))) return hipErrorInvalidValue;
  hipLaunchKernelGGL(rmsnorm_kernel, dim3((unsigned)rows), dim3(256), 0, stream, x, x_stride, gamma, out, cols, eps, planes);
  return hipGetLastError();
}

hipError_t launch_dyn_tanh(const float *x, long long x_stride, const float *gamma, const float *beta, float alpha,
                           float *out, int rows, int cols, hipStream_t stream, bool planes) {
  if (!x || !gamma || !beta || !out || rows < 1 || cols < 1 || x_stride < cols || (cols + 1023) / 1024 > 65535 ||
      (planes && (cols % 32 || x_stride % 4)))
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(dyn_tanh_kernel, dim3((unsigned)rows, (unsigned)((cols + 1023) / 1024)), dim3(256), 0, stream, x,
                     x_stride, gamma, beta, alpha, out, cols, planes);
  return hipGetLastError();
}

hipError_t launch_gather_rows(const float *x, const int *rows, float *out, int n, int cols, hipStream_t stream) {
  if (!x || !rows || !out || n < 1 || cols < 1) return hipErrorInvalidValue;
  // (a row gather is what the embedding lookup is)
  hipLaunchKernelGGL(embed_kernel, dim3((unsigned)n), dim3(256), 0, stream, x, rows, out, cols, 1.f,
                     (const float *)nullptr);
  return hipGetLastError();
}

hipError_t launch_add(const float *a, const float *b, float *out, long long n, hipStream_t stream) {
  if (n < 1) return hipErrorInvalidValue;
  const long long blocks = (n + 1023) / 1024;
  if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  hipLaunchKernelGGL(add_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, a, b, out, n);
  return hipGetLastError();
}

hipError_t launch_copy_floats(const float *x, float *out, long long n, hipStream_t stream) {
  if (!x || !out || n < 1 || (n + 1023) / 1024 > 0x7fffffffLL) return hipErrorInvalidValue;
  hipLaunchKernelGGL(copy_floats_kernel, dim3((unsigned)((n + 1023) / 1024)), dim3(256), 0, stream, x, out, n);
  return hipGetLastError();
}

hipError_t launch_swiglu_act(const float *gate_up, float *hidden, int rows, int ff, hipStream_t stream) {
  if (rows < 1 || rows > 65535 || ff < 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(swiglu_act_kernel, dim3((unsigned)((ff + 1023) / 1024), (unsigned)rows), dim3(256), 0, stream,
                     gate_up, hidden, ff);
  return hipGetLastError();
}

hipError_t launch_embed(const float *table, const int *tokens, float *out, int n_tokens, int d_model,
                        hipStream_t stream, float scale, const float *positions) {
  if (n_tokens < 1 || d_model < 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(embed_kernel, dim3((unsigned)n_tokens), dim3(256), 0, stream, table, tokens, out, d_model, scale,
                     positions);
  return hipGetLastError();
}

hipError_t launch_embed_list(const float *table, const IdList &tokens, float *out, int n_tokens, int d_model,
                             hipStream_t stream, float scale, const float *positions) {
  if (n_tokens < 1 || n_tokens > kIdList || d_model < 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(embed_list_kernel, dim3((unsigned)n_tokens), dim3(256), 0, stream, table, tokens, out, d_model, scale,
                     positions);
  return hipGetLastError();
}

hipError_t launch_add_bias_row(float *logits, const float *bias, int n, hipStream_t stream) {
  if (n < 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(add_bias_row_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, logits, bias, n);
  return hipGetLastError();
}

hipError_t launch_repetition_penalty(float *logits, int vocab, const int *ids, int n, double penalty,
                                     hipStream_t stream) {
  if (n < 1) return hipSuccess;
  hipLaunchKernelGGL(repetition_penalty_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, logits, vocab, ids, n,
                     penalty);
  return hipGetLastError();
}

hipError_t launch_repetition_penalty_list(float *logits, int vocab, const IdList &ids, int n, double penalty,
                                          hipStream_t stream) {
  if (n < 1) return hipSuccess;
  if (n > kIdList) return hipErrorInvalidValue;
  hipLaunchKernelGGL(repetition_penalty_list_kernel, dim3(1), dim3(256), 0, stream, logits, vocab, ids, n, penalty);
  return hipGetLastError();
}

hipError_t launch_rope_apply(const float *x, float *out, int seq_len, int head_dim, int start_pos, double theta,
                             hipStream_t stream) {
  if (!x || !out || seq_len < 0 || head_dim < 1) return hipErrorInvalidValue;
  const long long items = (long long)seq_len * (head_dim / 2 + (head_dim & 1));
  if (items == 0) return hipSuccess;
  if ((items + 255) / 256 > 0x7fffffffLL) return hipErrorInvalidValue;
  hipLaunchKernelGGL(rope_apply_kernel, dim3((unsigned)((items + 255) / 256)), dim3(256), 0, stream, x, out, seq_len,
                     head_dim, start_pos, theta);
  return hipGetLastError();
}

size_t topk_scratch_bytes(int vocab, int k) {
  return (size_t)((vocab + kTopkChunk - 1) / kTopkChunk) * k * sizeof(unsigned long long);
}

hipError_t launch_topk(const float *logits, int vocab, int k, bool finite_only, void *scratch, int *out_ids,
                       float *out_vals, int *out_count, hipStream_t stream, int fallback_id, int *pick, double temperature,
                       double r) {
  if (vocab < 1 || k < 1 || k > kMaxTopK || !scratch || (pick && !(temperature > 0.0))) return hipErrorInvalidValue;
  const int chunks = (vocab + kTopkChunk - 1) / kTopkChunk;
  unsigned long long *cand = (unsigned long long *)scratch;
  hipLaunchKernelGGL(topk_chunk_kernel, dim3((unsigned)chunks), dim3(kTopkThreads), 0, stream, logits, vocab, k,
                     finite_only ? 1 : 0, cand);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(topk_merge_kernel, dim3(1), dim3(kTopkThreads), 0, stream, logits, cand, chunks * k, k, out_ids, out_vals,
                     out_count, fallback_id, pick, temperature, r);
  return hipGetLastError();
}

hipError_t launch_greedy_embed(const float *logits, int vocab, void *scratch, int *id, const float *table, float *out, int d_model,
                               float scale, const float *position, hipStream_t stream) {
  if (!logits || vocab < 1 || !scratch || !id || !table || !out || d_model < 1) return hipErrorInvalidValue;
  unsigned long long *cand = nullptr;
  int chunks = 0;
  if (vocab > 65536) {
    chunks = (vocab + kTopkChunk - 1) / kTopkChunk;
    cand = (unsigned long long *)scratch;
    hipLaunchKernelGGL(topk_chunk_kernel, dim3((unsigned)chunks), dim3(kTopkThreads), 0, stream, logits, vocab, 1, 1, cand);
    if (const hipError_t e = hipGetLastError(); e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(greedy_embed_kernel, dim3(1), dim3(1024), 0, stream, logits, vocab, (const unsigned long long *)cand, chunks, id,
                     table, out, d_model, scale, position);
  return hipGetLastError();
}

}  // namespace shainet
