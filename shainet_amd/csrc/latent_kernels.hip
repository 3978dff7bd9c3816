// Latent attention on gfx950 (latent_kernels.hpp says what is computed), fp32.
//
// Decode is the absorbed form: per layer one launch that takes the queries to the latent space and
// appends the new rows, one that attends over key ranges in parallel, one that merges the ranges and
// takes the result back through W_uv; one row over few keys is a single launch (latent_row_kernel).  All heads share a cached row, so 16 (row, head) pairs are the
// columns of one MFMA tile and a row is read once per 16 of them.
//
// MFMA 16x16x4 layout (lane l): A[m = l % 16][k = l / 16], B[k = l / 16][n = l % 16],
// D[m = 4 (l / 16) + r][n = l % 16] for accumulator register r.  The contraction index may be
// visited in any order as long as A and B agree.
//
// Prefill is the expanded form: latent_prefill_kernel, split bf16 MFMA 32x32x16 over keys and values that a
// product made from the cached rows, the rotated key part read from the rows themselves.
#include "latent_kernels.hpp"
#include "split_mfma.hpp"

#include <math.h>
#include <stdint.h>
#include <stdlib.h>

namespace shainet {

namespace {

constexpr float kLog2e = 1.4426950408889634f;

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float sigmoid1(float z) { return 1.f / (1.f + expf(-z)); }

// element i of a rotated vector v of rot_dims turning elements
__device__ __forceinline__ float rotated(const float *v, int i, int rot_dims, const float2 *tab) {
  if (i >= rot_dims) return v[i];
  const float2 cs = tab[i >> 1];
  return (i & 1) ? v[i] * cs.x + v[i - 1] * cs.y : v[i] * cs.x - v[i + 1] * cs.y;
}

// One new row: 256 threads.
__device__ __forceinline__ void append_row(const LatentRows &r, const LatentShape &sh, int t) {
  __shared__ double red[4];
  const float *raw = r.raw + (long long)t * r.stride + r.kv_off;
  float *dst = r.rows + (long long)(r.start_row + t) * sh.row_w;
  double sq = 0.0;
  for (int i = threadIdx.x; i < sh.kv_rank; i += 256) sq += (double)raw[i] * (double)raw[i];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) sq += __shfl_xor(sq, o);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sq;
  __syncthreads();
  const double rms = sqrt(((red[0] + red[1]) + (red[2] + red[3])) / (double)sh.kv_rank + r.eps);
  const float2 *tab = r.rope_tab + (long long)(r.start_pos + t) * (sh.rot_dims >> 1);
  for (int i = threadIdx.x; i < sh.row_w; i += 256) {
    float v = 0.f;
    if (i < sh.kv_rank)
      v = (float)(((double)raw[i] / rms) * (double)r.kv_norm[i]);
    else if (i < sh.kv_rank + sh.rot_dim)
      v = rotated(raw + sh.kv_rank, i - sh.kv_rank, sh.rot_dims, tab);
    dst[i] = v;
  }
}

// q (nullable): the rotated parts of the row's queries turn in place
__global__ __launch_bounds__(256) void latent_append_kernel(LatentRows r, LatentShape sh, float *q) {
  append_row(r, sh, blockIdx.x);
  const int half = sh.rot_dims >> 1;
  if (!q || half == 0) return;
  const int qd = sh.dim + sh.rot_dim;
  float *qt = q + (long long)blockIdx.x * sh.H * qd + sh.dim;
  const float2 *tab = r.rope_tab + (long long)(r.start_pos + blockIdx.x) * half;
  for (int i = threadIdx.x; i < sh.H * half; i += 256) {
    const int h = i / half, p = i - h * half;
    float *v = qt + (long long)h * qd + 2 * p;
    const float x = v[0], y = v[1];
    const float2 cs = tab[p];
    v[0] = x * cs.x - y * cs.y;
    v[1] = y * cs.x + x * cs.y;
  }
}

// Workgroups 0 .. T - 1 append a row each; the others take 64 columns of one head of RT rows: lane =
// column, the wavefronts share the head's `dim` rows of W_uk and add up through LDS.
template <int RT>
__global__ __launch_bounds__(256) void latent_absorb_kernel(const float *__restrict__ q, const float *__restrict__ uk,
                                                            LatentRows r, LatentShape sh, int T,
                                                            float *__restrict__ q_abs, float qscale) {
  extern __shared__ float smem[];  // [RT][dim] query rows, then [4][RT][64] sums
  if ((int)blockIdx.x < T) {
    append_row(r, sh, blockIdx.x);
    return;
  }
  const int col_tiles = (sh.kv_rank + 63) / 64;
  int w = (int)blockIdx.x - T;
  const int ct = w % col_tiles;
  w /= col_tiles;
  const int h = w % sh.H, t0 = w / sh.H * RT;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int qd = sh.dim + sh.rot_dim;
  const int nt = min(RT, T - t0);
  const float *qh = q + ((long long)t0 * sh.H + h) * qd;
  const int col = ct * 64 + lane;
  const int per = (sh.dim + 3) / 4, d0 = wave * per, d1 = min(sh.dim, d0 + per);
  const float *wp = uk + (long long)h * sh.dim * sh.kv_rank + min(col, sh.kv_rank - 1);
  // the first rows of W_uk are on their way while the queries are staged
  constexpr int U = 16;
  float wv[U];
#pragma unroll
  for (int u = 0; u < U; ++u) wv[u] = wp[(long long)min(d0 + u, sh.dim - 1) * sh.kv_rank];
  for (int i = threadIdx.x; i < RT * sh.dim; i += 256) {
    const int rr = i / sh.dim, d = i - rr * sh.dim;
    smem[i] = rr < nt ? qh[(long long)rr * sh.H * qd + d] : 0.f;
  }
  __syncthreads();
  float acc[RT];
#pragma unroll
  for (int a = 0; a < RT; ++a) acc[a] = 0.f;
  for (int db = d0; db < d1; db += U) {
    if (db > d0) {
#pragma unroll
      for (int u = 0; u < U; ++u) wv[u] = wp[(long long)min(db + u, sh.dim - 1) * sh.kv_rank];
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (db + u < d1) {
#pragma unroll
        for (int a = 0; a < RT; ++a) acc[a] += smem[a * sh.dim + db + u] * wv[u];
      }
  }
  float *red = smem + RT * sh.dim;
#pragma unroll
  for (int a = 0; a < RT; ++a) red[(wave * RT + a) * 64 + lane] = acc[a];
  __syncthreads();
  for (int i = threadIdx.x; i < nt * 64; i += 256) {
    const int a = i >> 6, c = i & 63, cc = ct * 64 + c;
    if (cc >= sh.kv_rank) continue;
    const float s = (red[(0 * RT + a) * 64 + c] + red[(1 * RT + a) * 64 + c]) +
                    (red[(2 * RT + a) * 64 + c] + red[(3 * RT + a) * 64 + c]);
    q_abs[((long long)(t0 + a) * sh.H + h) * sh.row_w + cc] = s * qscale;
  }
  if (ct == 0) {  // the rotated part and the padding of these rows
    const int tail = sh.row_w - sh.kv_rank;
    for (int i = threadIdx.x; i < nt * tail; i += 256) {
      const int a = i / tail, e = i - a * tail;
      float v = 0.f;
      if (e < sh.rot_dim)
        v = rotated(qh + (long long)a * sh.H * qd + sh.dim, e, sh.rot_dims,
                    r.rope_tab + (long long)(r.start_pos + t0 + a) * (sh.rot_dims >> 1)) * qscale;
      q_abs[((long long)(t0 + a) * sh.H + h) * sh.row_w + sh.kv_rank + e] = v;
    }
  }
}

// Column c of tile ct is (row, head) pair 16 ct + c = row * H + head.  The workgroup (eight wavefronts)
// walks its share of the tile's keys in steps of KT: the cached rows go to LDS once and serve as keys
// (the scores' contraction is shared between the wavefronts) and as values (the wavefronts share the
// columns of the output, NTW tiles of 16 each).  Everything the first step needs is requested at
// once and the next step's rows while this one's are used: a launch of one new row is one step or two
// per workgroup, bound by its memory round trips.  Row stride row_w + 4 in LDS: 16-byte reads down a
// column of rows, and reads of 16 neighbours in rows 4 j apart, touch every bank once.
template <int KT, int NTW>
__global__ __launch_bounds__(512) void latent_absorbed_kernel(const float *__restrict__ q_abs,
                                                              const float *__restrict__ rows,
                                                              float *__restrict__ part_o, float *__restrict__ part_ml,
                                                              LatentShape sh, int T, int start_row, int splits,
                                                              int tiles_per_split, int v_w) {
  constexpr int NTH = 512, SUB = KT / 16, PARTS = 8 / SUB;
  constexpr int TPR = NTH / KT;                          // threads per key row; 32 per query row
  constexpr int UK = KT == 32 ? 13 : 10, UQ = KT == 32 ? 7 : 10;  // 16-byte pieces per thread: the widest rows plan_latent_absorbed admits
  extern __shared__ __attribute__((aligned(16))) float smem[];
  const int row_w = sh.row_w, ldr = row_w + 4;
  float *qs = smem, *ks = qs + 16 * ldr, *ss = ks + KT * ldr;  // ss: [PARTS][KT][17]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 15, j = lane >> 4;
  const int ct = blockIdx.x, sp = blockIdx.y, d_first = blockIdx.z * 1024;
  const int pairs = T * sh.H, v0 = ct * 16, v1 = min(v0 + 15, pairs - 1);
  const int lo = sh.window ? max(0, start_row + v0 / sh.H - sh.window + 1) : 0, hi = start_row + v1 / sh.H;
  const int my = min(v0 + n, pairs - 1), my_pos = start_row + my / sh.H;
  const int my_lo = sh.window ? max(0, my_pos - sh.window + 1) : 0;
  const int n_tiles = (hi - lo) / KT + 1;
  const int tile0 = sp * tiles_per_split, tile1 = min(n_tiles, tile0 + tiles_per_split);
  const int w4 = row_w >> 2;

  // a thread's pieces of its row: sub, sub + TPR, ... (past the end: the last one again, to the same place);
  // rows past the last key repeat it
  const int krow = threadIdx.x / TPR, ksub = threadIdx.x % TPR, qrow = threadIdx.x >> 5, qsub = threadIdx.x & 31;
  f32x4 kv[UK];
  auto load_keys = [&](int tile) {
    const float *src = rows + (long long)min(lo + tile * KT + krow, hi) * row_w;
#pragma unroll
    for (int u = 0; u < UK; ++u)
      if (TPR * u < w4) kv[u] = *(const f32x4 *)(src + 4 * min(ksub + TPR * u, w4 - 1));
  };
  auto park_keys = [&]() {
#pragma unroll
    for (int u = 0; u < UK; ++u)
      if (TPR * u < w4) *(f32x4 *)(ks + krow * ldr + 4 * min(ksub + TPR * u, w4 - 1)) = kv[u];
  };

  float m = -INFINITY, l = 0.f;
  f32x4 acc[NTW];
#pragma unroll
  for (int i = 0; i < NTW; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (tile0 < tile1) {
    f32x4 qv[UQ];
    const float *src = q_abs + (long long)min(v0 + qrow, v1) * row_w;
#pragma unroll
    for (int u = 0; u < UQ; ++u)
      if (32 * u < w4) qv[u] = *(const f32x4 *)(src + 4 * min(qsub + 32 * u, w4 - 1));
    load_keys(tile0);
#pragma unroll
    for (int u = 0; u < UQ; ++u)
      if (32 * u < w4) *(f32x4 *)(qs + qrow * ldr + 4 * min(qsub + 32 * u, w4 - 1)) = qv[u];
  }
  const int sub = wave % SUB, part = wave / SUB;
  const int steps = row_w >> 4, s_begin = part * steps / PARTS, s_end = (part + 1) * steps / PARTS;
  const int v_tiles = min((v_w - d_first) >> 4, 64);
  for (int tile = tile0; tile < tile1; ++tile) {
    const int k0 = lo + tile * KT;
    park_keys();
    if (tile + 1 < tile1) load_keys(tile + 1);
    __syncthreads();
    {
      f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
      const float *kp = ks + (16 * sub + n) * ldr + 4 * j, *qp = qs + n * ldr + 4 * j;
      // (fragments two steps ahead of the MFMAs that use them; the reads past the end stay inside LDS)
      f32x4 a1 = *(const f32x4 *)(kp + 16 * s_begin), b1 = *(const f32x4 *)(qp + 16 * s_begin);
      f32x4 a2 = *(const f32x4 *)(kp + 16 * min(s_begin + 1, steps - 1)), b2 = *(const f32x4 *)(qp + 16 * min(s_begin + 1, steps - 1));
      for (int i = s_begin; i < s_end; ++i) {
        const f32x4 a = a1, b = b1;
        const int ahead = min(i + 2, steps - 1);
        a1 = a2;
        b1 = b2;
        a2 = *(const f32x4 *)(kp + 16 * ahead);
        b2 = *(const f32x4 *)(qp + 16 * ahead);
        s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, s1, 0, 0, 0);
        s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, s1, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) ss[(part * KT + 16 * sub + 4 * j + r) * 17 + n] = s0[r] + s1[r];
    }
    __syncthreads();
    // every wavefront: the whole tile's scores of its columns, key 16 u + 4 j + r in p[u][r]
    float p[SUB][4], mx = -INFINITY;
#pragma unroll
    for (int u = 0; u < SUB; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int kk = 16 * u + 4 * j + r;
        float s = ss[kk * 17 + n];
#pragma unroll
        for (int g = 1; g < PARTS; ++g) s += ss[(g * KT + kk) * 17 + n];
        const int key = k0 + kk;
        p[u][r] = key >= my_lo && key <= my_pos ? s : -INFINITY;
        mx = fmaxf(mx, p[u][r]);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16));
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float mnew = fmaxf(m, mx);
    const float mref = mnew == -INFINITY ? 0.f : mnew;  // no key of this column seen so far
    const float alpha = fast_exp2(m - mref);
    float ps = 0.f;
#pragma unroll
    for (int u = 0; u < SUB; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        p[u][r] = fast_exp2(p[u][r] - mref);
        ps += p[u][r];
      }
    l = l * alpha + ps;
    m = mnew;
#pragma unroll
    for (int i = 0; i < NTW; ++i) acc[i] *= alpha;
#pragma unroll
    for (int i = 0; i < NTW; ++i) {
      // (a wavefront without an i-th tile computes the last one again and does not store it)
      const float *vp = ks + 4 * j * ldr + d_first + 16 * min(wave + 8 * i, v_tiles - 1) + n;
#pragma unroll
      for (int u = 0; u < SUB; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(vp[(16 * u + r) * ldr], p[u][r], acc[i], 0, 0, 0);
    }
    __syncthreads();  // the rows are free for the next step's
  }
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);
  const long long slot = (long long)(v0 + n) * splits + sp;
#pragma unroll
  for (int i = 0; i < NTW; ++i) {
    const int vt = wave + 8 * i;
    if (vt < v_tiles) *(f32x4 *)(part_o + slot * v_w + d_first + 16 * vt + 4 * j) = acc[i];
  }
  if (wave == 0 && j == 0 && blockIdx.z == 0) *(float2 *)(part_ml + 2 * slot) = float2{m, l};
}

// Sixteen outputs of one head, a wavefront each, for RT rows.  blockIdx.x: head fastest, so that with
// a multiple of 8 heads the workgroups that merge the same partials sit on one XCD; blockIdx.y: rows.
// The wavefronts' rows of W_uv and the partials are requested before anything is waited for.
template <int RT>
__global__ __launch_bounds__(1024) void latent_out_kernel(const float *__restrict__ part_o,
                                                          const float *__restrict__ part_ml,
                                                          const float *__restrict__ uv, const float *__restrict__ sink,
                                                          LatentRows r, LatentShape sh, int T, int splits, int v_w,
                                                          float *__restrict__ out) {
  extern __shared__ __attribute__((aligned(16))) float smem[];
  constexpr int WU = 4;   // 16-byte pieces of a row of W_uv per lane held in registers
  constexpr int LD = 12;  // partials in flight per thread
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int h = blockIdx.x % sh.H, t0 = blockIdx.y * RT, nt = min(RT, T - t0);
  const int v4 = v_w >> 2, groups = 1024 / v4;  // thread: column of 16 bytes c, ranges g, g + groups, ...
  const int c = threadIdx.x % v4, g = threadIdx.x / v4;
  float *lat = smem, *fac = lat + RT * v_w, *red = fac + RT * splits;  // [RT][v_w], [RT][splits], [groups][v_w]
  const int jj = (int)(blockIdx.x / sh.H) * 16 + wave;
  const float *wr = uv + ((long long)h * sh.vdim + min(jj, sh.vdim - 1)) * sh.kv_rank;
  const bool held = (sh.kv_rank & 3) == 0 && sh.kv_rank <= 256 * WU;
  f32x4 w[WU];
  if (held) {
#pragma unroll
    for (int u = 0; u < WU; ++u)
      if (256 * u < sh.kv_rank) w[u] = *(const f32x4 *)(wr + min(256 * u + 4 * lane, sh.kv_rank - 4));
  }
  for (int a = 0; a < nt; ++a) {
    const long long col = (long long)(t0 + a) * sh.H + h;
    const float *po = part_o + col * splits * v_w + 4 * c;
    f32x4 x[LD];
#pragma unroll
    for (int u = 0; u < LD; ++u)
      if (groups * u < splits) x[u] = *(const f32x4 *)(po + (long long)min(g + groups * u, splits - 1) * v_w);
    // the factor of a range: 2^(max - overall max) / denominator, the sink included in both (an empty
    // range has max -inf and sum 0: factor 0)
    if (wave == 0) {
      const float2 *ml = (const float2 *)part_ml + col * splits;
      const float sk = sink[h] * kLog2e;
      float mm = sk;
      for (int s = lane; s < splits; s += 64) mm = fmaxf(mm, ml[s].x);
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) mm = fmaxf(mm, __shfl_xor(mm, o));
      float den = 0.f;
      for (int s = lane; s < splits; s += 64) den += ml[s].y * fast_exp2(ml[s].x - mm);
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) den += __shfl_xor(den, o);
      const float inv = 1.f / (den + fast_exp2(sk - mm));
      for (int s = lane; s < splits; s += 64) fac[a * splits + s] = fast_exp2(ml[s].x - mm) * inv;
    }
    __syncthreads();
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < LD; ++u)
      if (g + groups * u < splits) sum += fac[a * splits + g + groups * u] * x[u];
    for (int s = g + groups * LD; s < splits; s += groups) sum += fac[a * splits + s] * *(const f32x4 *)(po + (long long)s * v_w);
    if (g < groups) *(f32x4 *)(red + g * v_w + 4 * c) = sum;
    __syncthreads();
    for (int i = threadIdx.x; i < v_w; i += 1024) {
      float s = red[i];
      for (int k = 1; k < groups; ++k) s += red[k * v_w + i];
      lat[a * v_w + i] = s;
    }
    __syncthreads();
  }
  if (jj >= sh.vdim) return;
  float s[RT];
#pragma unroll
  for (int a = 0; a < RT; ++a) s[a] = 0.f;
  if (held) {
#pragma unroll
    for (int u = 0; u < WU; ++u)
      if (256 * u + 4 * lane < sh.kv_rank) {
#pragma unroll
        for (int a = 0; a < RT; ++a) {
          const f32x4 x = *(const f32x4 *)(lat + a * v_w + 256 * u + 4 * lane);
          s[a] += (w[u].x * x.x + w[u].y * x.y) + (w[u].z * x.z + w[u].w * x.w);
        }
      }
  } else {
    for (int k = lane; k < sh.kv_rank; k += 64) {
      const float wv = wr[k];
#pragma unroll
      for (int a = 0; a < RT; ++a) s[a] += wv * lat[a * v_w + k];
    }
  }
#pragma unroll
  for (int a = 0; a < RT; ++a) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s[a] += __shfl_xor(s[a], o);
    if (lane == 0 && a < nt)
      out[((long long)(t0 + a) * sh.H + h) * sh.vdim + jj] =
          s[a] * sigmoid1(r.raw[(long long)(t0 + a) * r.stride + r.gate_off + h]);
  }
}

// One new row that sees few keys: the append, the queries' way to the latent space, the attention and the way back in one
// launch, a workgroup of 512 threads per head.  A row (of the cache, W_uk or W_uv) is read by 16 lanes, P pieces of 16 bytes each,
// so that the 32 quarters of the wavefronts take 32 keys a round, G rounds in registers, of which a score needs a sum over
// 16 lanes and the weighted sum nothing more: keys are read once.  Each quarter keeps its own online softmax; quarters meet in
// registers, wavefronts in LDS.  Everything that the first rounds need is requested before anything is waited for.
// Bound by what a compute unit gets from its L2 (64 bytes a clock: 422 KB of 16 heads' share at 180 keys), whose way is kept
// for what is needed next: keys are requested behind W_uk, and W_uv behind the keys (all at once in front: 10.4 us), and by
// the meetings.  16 heads of 64 + 32 and 64 dimensions, latents of 256: us, three launches and the gaps between them | this:
// 30 keys 18.0 | 7.5, 110 keys 17.8 | 7.6, 190 keys 18.8 | 8.7, 410 keys 18.8 | 12.5, 810 keys 18.9 | 16.8; of 128 + 64 and 128,
// latents of 512: 30 keys 21.0 | 12.0, 190 keys 21.5 | 16.3, 410 keys 21.6 | 20.5.
template <int CTRL>
__device__ __forceinline__ float dpp(float x) { return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, false)); }
template <int CTRL>
__device__ __forceinline__ double dpp(double x) {
  return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xf, 0xf, false),
                          __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xf, 0xf, false));
}
// the sum over 16 neighbouring lanes, in each of them (rotations by 8, 4, 2 and 1)
template <class V>
__device__ __forceinline__ V sum16(V x) {
  x += dpp<0x128>(x);
  x += dpp<0x124>(x);
  x += dpp<0x122>(x);
  return x + dpp<0x121>(x);
}
// lane l's value and that of the same lane of the other quarter of its half (WIDE: of the other half)
template <bool WIDE>
__device__ __forceinline__ float2 both(float x) {
  const unsigned b = __float_as_uint(x);
  typedef unsigned pair_t __attribute__((ext_vector_type(2)));
  pair_t r;
  if constexpr (WIDE)
    r = __builtin_amdgcn_permlane32_swap(b, b, false, false);
  else
    r = __builtin_amdgcn_permlane16_swap(b, b, false, false);
  return float2{__uint_as_float(r.x), __uint_as_float(r.y)};
}
__device__ __forceinline__ float sum_quarters(float x) {
  float2 v = both<false>(x);
  v = both<true>(v.x + v.y);
  return v.x + v.y;
}
__device__ __forceinline__ float max_quarters(float x) {
  float2 v = both<false>(x);
  v = both<true>(fmaxf(v.x, v.y));
  return fmaxf(v.x, v.y);
}

template <int P>
struct RowPieces {
  f32x4 x[P];
  // a row of a base that all threads share; at: where the lane's pieces lie in a row
  __device__ __forceinline__ void request(const float *base, unsigned row, const unsigned (&at)[P]) {
#pragma unroll
    for (int u = 0; u < P; ++u) x[u] = *(const f32x4 *)((const char *)base + (row + at[u]));
  }
  __device__ __forceinline__ float dot(const f32x4 (&y)[P]) const {  // in all 16 lanes
    float s = 0.f, t = 0.f;
#pragma unroll
    for (int u = 0; u < P; ++u) {
      s = fmaf(x[u].x, y[u].x, fmaf(x[u].y, y[u].y, s));
      t = fmaf(x[u].z, y[u].z, fmaf(x[u].w, y[u].w, t));
    }
    return sum16(s + t);
  }
};

template <int P, int G, int RK, int RV>
__global__ __launch_bounds__(512) void latent_row_kernel(const float *__restrict__ q, const float *__restrict__ uk,
                                                         const float *__restrict__ uv, const float *__restrict__ sink, LatentRows r,
                                                         LatentShape sh, float qscale, float *__restrict__ out) {
  constexpr int W4 = 16 * P, kOwn = (64 * P + 511) / 512;
  __shared__ f32x4 part[8][W4], qa[128 * kOwn], fresh[128 * kOwn];
  __shared__ float top[8], sums[8];
  const int h = blockIdx.x, tid = threadIdx.x, lane = tid & 63, l = tid & 15, quarter = tid >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int w4 = sh.row_w >> 2, k4 = sh.kv_rank >> 2, dim = sh.dim, vdim = sh.vdim, half = sh.rot_dims >> 1;
  const int lo = sh.window ? max(0, r.start_row - sh.window + 1) : 0, n_old = r.start_row - lo;
  const float *const qh = q + (long long)h * (dim + sh.rot_dim);
  const float *const ukh = uk + (long long)h * dim * sh.kv_rank, *const uvh = uv + (long long)h * vdim * sh.kv_rank;
  const float *const raw = r.raw + r.kv_off, *const keys = r.rows + (long long)lo * sh.row_w;
  const unsigned k_bytes = 4u * sh.kv_rank, row_bytes = 4u * sh.row_w;
  unsigned at_k[P], at_row[P];  // (past the end: the last piece again)
#pragma unroll
  for (int u = 0; u < P; ++u) {
    at_k[u] = 16u * min(l + 16 * u, k4 - 1);
    at_row[u] = 16u * min(l + 16 * u, w4 - 1);
  }

  // what the new row and the rotated queries are made of: elements tid, tid + 512, ...
  float squares[P], from[kOwn], beside[kOwn], q_from[kOwn], q_beside[kOwn], gamma[kOwn];
  float2 turn[kOwn];
#pragma unroll
  for (int u = 0; u < P; ++u) squares[u] = raw[min(lane + 64 * u, sh.kv_rank - 1)];
#pragma unroll
  for (int u = 0; u < kOwn; ++u) {
    const int i = min(tid + 512 * u, sh.kv_rank + sh.rot_dim - 1), e = i - sh.kv_rank;
    const bool turns = e >= 0 && e < sh.rot_dims;
    from[u] = raw[i];
    beside[u] = raw[turns ? sh.kv_rank + (e ^ 1) : i];
    q_from[u] = qh[e >= 0 ? dim + e : 0];
    q_beside[u] = qh[turns ? dim + (e ^ 1) : 0];
    gamma[u] = r.kv_norm[min(i, sh.kv_rank - 1)];
    turn[u] = float2{1.f, 0.f};
    if (half) turn[u] = r.rope_tab[(long long)r.start_pos * half + (turns ? e >> 1 : 0)];
  }
  const float gate = r.raw[r.gate_off + h], sk = sink[h] * kLog2e;

  RowPieces<P> w[RK];
  float qd[RK];
  auto load_uk = [&](int i, int d) {
    w[i].request(ukh, min(d, dim - 1) * k_bytes, at_k);
    qd[i] = qh[min(d, dim - 1)];
  };
#pragma unroll
  for (int i = 0; i < RK; ++i) load_uk(i, quarter + 32 * i);
  __builtin_amdgcn_sched_barrier(0);

  // the new row
  double sq = 0.0;
#pragma unroll
  for (int u = 0; u < P; ++u) sq += lane + 64 * u < sh.kv_rank ? (double)squares[u] * (double)squares[u] : 0.0;
  sq = sum16(sq);
  sq += __shfl_xor(sq, 16);
  sq += __shfl_xor(sq, 32);
  const double rms = sqrt(sq / (double)sh.kv_rank + r.eps);
#pragma unroll
  for (int u = 0; u < kOwn; ++u) {
    const int i = tid + 512 * u, e = i - sh.kv_rank;
    const bool turns = e < sh.rot_dims, inside = e < sh.rot_dim;
    const float c = turns ? turn[u].x : 1.f, s = !turns ? 0.f : (e & 1) ? turn[u].y : -turn[u].y;
    const float normed = (float)(((double)from[u] / rms) * (double)gamma[u]);
    const float v = e < 0 ? normed : !inside ? 0.f : turns ? from[u] * c + beside[u] * s : from[u];
    ((float *)fresh)[i] = v;
    if (h == 0 && i < sh.row_w) r.rows[(long long)r.start_row * sh.row_w + i] = v;
    ((float *)qa)[i] = !inside ? 0.f : (turns ? q_from[u] * c + q_beside[u] * s : q_from[u]) * qscale;
  }

  // the queries' way to the latent space
  f32x4 acc[P];
#pragma unroll
  for (int u = 0; u < P; ++u) acc[u] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto take_uk = [&](int d) {
#pragma unroll
    for (int i = 0; i < RK; ++i) {
      const float x = d + 32 * i < dim ? qd[i] : 0.f;
#pragma unroll
      for (int u = 0; u < P; ++u) acc[u] += x * w[i].x[u];
    }
  };
  take_uk(quarter);  // (what is in flight for later is not waited for here, as it would be in the loop)
  for (int d = quarter + 32 * RK; d - quarter < dim; d += 32 * RK) {
#pragma unroll
    for (int i = 0; i < RK; ++i) load_uk(i, d + 32 * i);
    take_uk(d);
  }
  // keys k0 .. k0 + 32 G - 1, those that there are (a wavefront without any asks for none: a compute unit's way to its L2 is what
  // the launch waits for)
  RowPieces<P> kv[G];
  auto load_keys = [&](int k0) {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (k0 + 32 * g + 4 * wave < n_old) {
        kv[g].request(keys, min(k0 + 32 * g + quarter, n_old - 1) * row_bytes, at_row);
      } else {
#pragma unroll
        for (int u = 0; u < P; ++u) kv[g].x[u] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
    }
  };
  __builtin_amdgcn_sched_barrier(0);
  load_keys(0);
  __builtin_amdgcn_sched_barrier(0);
  auto meet = [&]() {  // acc of the quarters of a wavefront
#pragma unroll
    for (int u = 0; u < P; ++u) {
      f32x4 t;
#pragma unroll
      for (int e = 0; e < 4; ++e) t[e] = sum_quarters(acc[u][e]);
      if (lane < 16) part[wave][l + 16 * u] = t;
    }
  };
  meet();
  __syncthreads();
  if (tid < k4) {
    f32x4 t[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) t[i] = part[i][tid];
    qa[tid] = (((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]))) * qscale;
  }
  __syncthreads();

  // quarter 0 begins with the new row, the others with none
  RowPieces<P> own;
  f32x4 qv[P];
#pragma unroll
  for (int u = 0; u < P; ++u) {
    qv[u] = qa[l + 16 * u];
    own.x[u] = fresh[l + 16 * u];
  }
  float m = own.dot(qv), den = 1.f;
  if (quarter > 0) m = -INFINITY, den = 0.f;
#pragma unroll
  for (int u = 0; u < P; ++u) acc[u] = quarter > 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : own.x[u];
  auto attend = [&](int k0) {
    float s[G], most = m;
#pragma unroll
    for (int g = 0; g < G; ++g) {
#pragma unroll
      for (int u = 0; u < P; ++u)
        if (16 * u + 15 >= w4) kv[g].x[u] = l + 16 * u < w4 ? kv[g].x[u] : f32x4{0.f, 0.f, 0.f, 0.f};
      s[g] = kv[g].dot(qv);
      if (k0 + 32 * g + quarter >= n_old) s[g] = -INFINITY;
      most = fmaxf(most, s[g]);
    }
    const float ref = most == -INFINITY ? 0.f : most;  // no key seen so far
    const float alpha = fast_exp2(m - ref);
    m = most;
    den *= alpha;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      s[g] = fast_exp2(s[g] - ref);
      den += s[g];
    }
#pragma unroll
    for (int u = 0; u < P; ++u) {
      acc[u] *= alpha;
#pragma unroll
      for (int g = 0; g < G; ++g) acc[u] += s[g] * kv[g].x[u];
    }
  };
  attend(0);
  for (int k0 = 32 * G; k0 < n_old; k0 += 32 * G) {
    load_keys(k0);
    attend(k0);
  }
  // (W_uv behind the keys: what else is on its way holds them up)
  RowPieces<P> v[RV];
  auto load_uv = [&](int i, int j) { v[i].request(uvh, min(j, vdim - 1) * k_bytes, at_k); };
#pragma unroll
  for (int i = 0; i < RV; ++i) load_uv(i, quarter + 32 * i);
  __builtin_amdgcn_sched_barrier(0);

  const float wave_top = max_quarters(m), scale = fast_exp2(m - (wave_top == -INFINITY ? 0.f : wave_top));
#pragma unroll
  for (int u = 0; u < P; ++u) acc[u] *= scale;
  meet();
  den = sum_quarters(den * scale);
  if (lane == 0) {
    top[wave] = wave_top;
    sums[wave] = den;
  }
  __syncthreads();
  float mm = sk, all = 0.f, f[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) mm = fmaxf(mm, top[i]);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    f[i] = fast_exp2(top[i] - mm);
    all += f[i] * sums[i];
  }
  const float factor = sigmoid1(gate) / (all + fast_exp2(sk - mm));
  if (tid < k4) {
    f32x4 t[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) t[i] = part[i][tid] * f[i];
    qa[tid] = ((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]));
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < P; ++u) {
    qv[u] = qa[l + 16 * u];
    if (16 * u + 15 >= k4) qv[u] = l + 16 * u < k4 ? qv[u] : f32x4{0.f, 0.f, 0.f, 0.f};
  }
  auto give = [&](int j) {
#pragma unroll
    for (int i = 0; i < RV; ++i) {
      const float s = v[i].dot(qv);
      if (l == 0 && j + 32 * i < vdim) out[(long long)h * vdim + j + 32 * i] = s * factor;
    }
  };
  give(quarter);
  for (int j = quarter + 32 * RV; j - quarter < vdim; j += 32 * RV) {
#pragma unroll
    for (int i = 0; i < RV; ++i) load_uv(i, j + 32 * i);
    give(j);
  }
}

// ---- expanded form -----------------------------------------------------------------------------
//
// A workgroup owns 128 rows of one head, a wavefront 32 of them; all walk the keys in tiles of 32 that
// go global memory -> registers -> split -> LDS (one stage of keys, one of values; the values travel behind the
// score MFMAs, the next tile's keys behind the others).  Two workgroups share a compute unit, so that one's barriers
// hide behind the other's MFMAs.  Queries, keys, values and probabilities are exact sums of three bf16 numbers
// (split_mfma.hpp); queries of more than 128 dimensions have no registers for their parts and are split
// again for every tile, beside the MFMAs.  S^T = K Q^T, so that the probabilities come out of the accumulator laid out as
// the B operand of O^T += V^T P^T:
//   scores:  m = key within the tile, n = row; step i of lane half j covers d = 16 i + 8 j + 0..7;
//            d runs over the unrotated dimensions, padded to a multiple of 8, then the rotated ones.
//   output:  tile t, m: d = NT m + t; step u of lane half j covers keys 16 u + 4 j + {0..3, 8..11}.
// LDS in units of 16 bytes: keys [part][octet of d][key], an octet 33 units; values [part][group 2 u + j of eight
// keys][column], column d at place d / NT of block d % NT, 36 units a block.
// Bound by registers (256 of them: two wavefronts per SIMD) and the splits beside the MFMAs: 2048 rows of 16 heads of 192 and 128
// dimensions 268 -> 208 us against v_mfma_f32_32x32x2_f32, whose cycles the vector ALU cannot use.  (Two fp16 numbers a query
// and key, three products a score and the queries' parts in registers took a third less, but such numbers leave out up to
// 2^-21 of a product.)
// NK: pieces of 8 query / key dimensions at most; NT: tiles of 32 value dimensions.
struct LatentPrefillArgs {
  const float *q;        // [T, H (dim + rot_dim)], rotated (launch_latent_append)
  const float *kv;       // [key rows, H dim + H vdim]
  const float *key_rot;  // rotated part of key row 0; rows row_w apart
  const float *sink;
  LatentRows r;          // raw (gates), rope_tab, start_pos
  LatentShape sh;
  float *out;            // [T, H vdim]
  float *part_o, *part_ml;  // splits > 1: [blocks][splits][128][32 NT], [..][128][2]
  int T, first_key;      // row t sees key rows .. first_key + t
  int items, splits;
  float c;               // scale * log2(e)
};

template <int NK, int NT>
__global__ __launch_bounds__(256, NK <= 24 ? 2 : 1) void latent_prefill_kernel(const LatentPrefillArgs a) {
  constexpr int VSTR = NT * 32, KS = NK / 2;  // columns of the output; MFMA steps of the scores
  constexpr int KU = (NK + 7) / 8, VU = NT / 2;  // per thread: octets of a tile's keys, eight rows of a column of its values
  constexpr int kOct = 33, kPartK = NK * kOct, kGroup = NT * 36, kPartV = 4 * kGroup;
  constexpr bool HELD = NK <= 16 && NK * NT <= 48;  // the parts of the query stay in registers
  __shared__ __attribute__((aligned(16))) u32x4 lds[3 * kPartK + 3 * kPartV];
  const LatentShape &sh = a.sh;
  // heads fastest: with a multiple of 8 heads an XCD (index % 8) keeps to its own heads' keys and
  // values; the blocks with the most keys start first
  const int h = blockIdx.x % sh.H;
  const int chunk = (blockIdx.x / sh.H) % a.splits;
  const int item = a.items - 1 - (int)(blockIdx.x / sh.H / a.splits);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 31, j = lane >> 5;
  const int dn = sh.dim, dr = sh.rot_dim, dn8 = (dn + 7) / 8 * 8;
  const int row0 = item * 128, w_row0 = row0 + wave * 32;
  const bool wave_active = w_row0 < a.T;
  const int my_row = min(w_row0 + n, a.T - 1);
  const int my_hi = a.first_key + my_row, my_lo = sh.window ? max(0, my_hi - sh.window + 1) : 0;
  const int w_first = min(w_row0, a.T - 1), w_last = min(w_row0 + 31, a.T - 1);
  const int w_hi_min = a.first_key + w_first, w_hi_max = a.first_key + w_last;
  const int w_lo_min = sh.window ? max(0, w_hi_min - sh.window + 1) : 0;
  const int w_lo_max = sh.window ? max(0, w_hi_max - sh.window + 1) : 0;
  const int b_hi = a.first_key + min(row0 + 127, a.T - 1);
  const int b_lo = sh.window ? max(0, a.first_key + row0 - sh.window + 1) : 0;
  const int kt_all0 = b_lo >> 5, n_tiles = (b_hi >> 5) + 1 - kt_all0;
  const int per_chunk = (n_tiles + a.splits - 1) / a.splits;
  const int kt0 = kt_all0 + chunk * per_chunk, kt1 = min(kt_all0 + n_tiles, kt0 + per_chunk);

  const unsigned kv_stride = (unsigned)(sh.H * (sh.dim + sh.vdim));
  // staging: a thread takes octets sub, sub + 8, ... of one key's row (those behind the last one repeat it) and eight
  // rows of one or two groups of a column of the values
  const int k_row = threadIdx.x >> 3, sub = threadIdx.x & 7;
  const float *k_src[KU];
  bool k_rot[KU], k_whole[KU];  // part of the rotated dimensions; the octet's second half lies within the key
#pragma unroll
  for (int u = 0; u < KU; ++u) {
    const int d = 8 * min(sub + 8 * u, NK - 1), e = d - dn8;
    k_rot[u] = e >= 0 && e < dr;  // behind both parts the query is zero, any of the key's values will do
    k_src[u] = k_rot[u] ? a.key_rot + e : a.kv + h * dn + (d < dn8 ? d : 0);
    k_whole[u] = k_rot[u] ? e + 4 < dr : d + 4 < dn;
  }
  const int v_col = threadIdx.x % VSTR, v_group = threadIdx.x / VSTR;
  const int v_row = 16 * (v_group >> 1) + 4 * (v_group & 1);  // and 16 further on for the second
  const int v_unit = 3 * kPartK + v_group * kGroup + v_col % NT * 36 + v_col / NT;
  const unsigned v_off = v_col < sh.vdim ? v_col : 0;  // (columns beyond are never stored)
  const float *v_src = a.kv + sh.H * dn + h * sh.vdim;
  f32x4 stage[2 * (KU > VU ? KU : VU)];
  auto load_k = [&](int kt) {
    const unsigned key = (unsigned)min(kt * 32 + k_row, b_hi);
#pragma unroll
    for (int u = 0; u < KU; ++u) {
      const float *p = k_src[u] + (unsigned long long)key * (k_rot[u] ? (unsigned)sh.row_w : kv_stride);
      stage[2 * u] = *(const f32x4 *)p;
      stage[2 * u + 1] = *(const f32x4 *)(p + (k_whole[u] ? 4 : 0));
    }
  };
  auto load_v = [&](int kt) {
    if (kt * 32 + 31 <= b_hi) {
      const float *p = v_src + (unsigned long long)(unsigned)(kt * 32) * kv_stride;
      const unsigned off = (unsigned)v_row * kv_stride + v_off;
#pragma unroll
      for (int u = 0; u < VU; ++u)
#pragma unroll
        for (int i = 0; i < 8; ++i)
          stage[2 * u + (i >> 2)][i & 3] = (p + (unsigned long long)(16 * u + (i & 3) + 8 * (i >> 2)) * kv_stride)[off];
    } else {
#pragma unroll
      for (int u = 0; u < VU; ++u)
#pragma unroll
        for (int i = 0; i < 8; ++i)
          stage[2 * u + (i >> 2)][i & 3] =
              v_src[(unsigned long long)(unsigned)min(kt * 32 + v_row + 16 * u + (i & 3) + 8 * (i >> 2), b_hi) * kv_stride + v_off];
    }
  };
  auto park = [&](int u, int unit, int part, float lift) {
    u32x4 hi, mid, lo;
    split_octet(stage[2 * u] * lift, stage[2 * u + 1] * lift, hi, mid, lo);
    lds[unit] = hi;
    lds[unit + part] = mid;
    lds[unit + 2 * part] = lo;
  };
  auto park_k = [&]() {
#pragma unroll
    for (int u = 0; u < KU; ++u) park(u, min(sub + 8 * u, NK - 1) * kOct + k_row, kPartK, 1.f);
  };
  auto park_v = [&]() {
#pragma unroll
    for (int u = 0; u < VU; ++u) park(u, v_unit + 2 * u * kGroup, kPartV, kLift);
  };
  if (kt0 < kt1) load_k(kt0);

  f32x4 qr[HELD ? 1 : KS][2];
  u32x4 qf[HELD ? KS : 1][3];
  const float *q_row = a.q + ((long long)my_row * sh.H + h) * (dn + dr);
  QueryRange range;
#pragma unroll
  for (int i = 0; i < KS; ++i) {
    f32x4 x[2];
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      const int d = 16 * i + 8 * j + 4 * w, e = d - dn8;
      x[w] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (d < dn || (e >= 0 && e < dr)) x[w] = *(const f32x4 *)(q_row + (d < dn ? d : dn + e));
      range.add(x[w]);
      x[w] *= a.c;
    }
    if constexpr (HELD)
      split_octet(x[0], x[1], qf[i][0], qf[i][1], qf[i][2]);
    else
      qr[i][0] = x[0], qr[i][1] = x[1];
  }
  const bool apart = __any(range.apart(a.c));  // some query of the wavefront needs its scores in fp32
  f32x16 o[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[t][r] = 0.f;
  float m = -INFINITY, l = 0.f;  // reference value of the row's exponentials (log2 units), this lane half's sum
  constexpr float kTau = 8.f;    // scores may exceed it by this much before it moves

  // Per tile: the values travel while the scores are computed, the next tile's keys while the values
  // are used; each set is parked in LDS behind a barrier that says its stage is free.
  if (kt0 < kt1) park_k();
  __syncthreads();
  for (int kt = kt0; kt < kt1; ++kt) {
    load_v(kt);
    const int k_first = kt * 32, k_last = k_first + 31;
    const bool visible = wave_active && k_first <= w_hi_max && k_last >= w_lo_min;
    f32x16 s;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = 0.f;
    if (visible) {
      const u32x4 *kl = lds + j * kOct + n;
#pragma unroll
      for (int i = 0; i < KS; ++i) {
        u32x4 kf[3];
#pragma unroll
        for (int w = 0; w < 3; ++w) kf[w] = kl[w * kPartK + 2 * i * kOct];
        if constexpr (!HELD) {
          asm volatile("" : "+v"(qr[i][0]), "+v"(qr[i][1]));  // (not moved out of the loop over the tiles)
          split_octet(qr[i][0], qr[i][1], qf[0][0], qf[0][1], qf[0][2]);
        }
#pragma unroll
        for (int w = 0; w < 6; ++w) s = mfma_bf16(kf[kPartA[w]], qf[HELD ? i : 0][kPartB[w]], s);
      }
      if (k_first < w_lo_max || k_last > w_hi_min) {  // an edge of some row's keys lies in the tile
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = k_first + 8 * (r >> 2) + 4 * j + (r & 3);
          if (key < my_lo || key > my_hi) s[r] = -INFINITY;
        }
      }
      float mx = s[0];
#pragma unroll
      for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      const bool move = mx > (m == -INFINITY ? -INFINITY : m + kTau);
      if (__builtin_amdgcn_ballot_w64(move) != 0) {
        const float mnew = move ? mx : m;
        const float alpha = move && m != -INFINITY ? fast_exp2(m - mnew) : 1.f;  // (nothing to rescale before a row's first key)
        m = mnew;
        l *= alpha;
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[t][r] *= alpha;
      }
      const float mref = m == -INFINITY ? 0.f : m;
      float psum = 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[r] = fast_exp2(s[r] - mref);
        psum += s[r];
      }
      l += psum;
    }
    park_v();
    __syncthreads();
    if (kt + 1 < kt1) load_k(kt + 1);
    if (visible) {
      const u32x4 *vl = lds + 3 * kPartK + j * kGroup + n;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        u32x4 pf[3];
        split_octet(f32x4{s[8 * u], s[8 * u + 1], s[8 * u + 2], s[8 * u + 3]},
                    f32x4{s[8 * u + 4], s[8 * u + 5], s[8 * u + 6], s[8 * u + 7]}, pf[0], pf[1], pf[2]);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          u32x4 vf[3];
#pragma unroll
          for (int w = 0; w < 3; ++w) vf[w] = vl[w * kPartV + 2 * u * kGroup + 36 * t];
#pragma unroll
          for (int w = 0; w < 6; ++w) o[t] = mfma_bf16(vf[kPartA[w]], pf[kPartB[w]], o[t]);
        }
      }
    }
    if (kt + 1 < kt1) park_k();
    __syncthreads();
  }

  // Results that are not finite come from operands that are not (or are infinite once lifted): the
  // wavefront takes its keys again in fp32, which says which.  2048 rows of a layer of 16 heads of 192 and 128 dimensions, NaN in
  // row 5: 5.5 ms with its copies against 3.2 without (key by key, one dimension at a time, it was 89).
  float probe = l * 0.f;
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) probe = fmaf(o[t][r], 0.f, probe);
  if (__builtin_expect(wave_active && (apart || __any(probe != 0.f)), 0)) {
    // (what a lane works on is found again from its number: kept for here it would cost the loop above registers)
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int n = tid & 31, j = (tid & 63) >> 5, my_row = min(w_row0 + n, a.T - 1);
    const int my_hi = a.first_key + my_row, my_lo = sh.window ? max(0, my_hi - sh.window + 1) : 0;
    const float *q_row = a.q + ((long long)my_row * sh.H + h) * (dn + dr), *v_src = a.kv + sh.H * dn + h * sh.vdim;
    f32x16 s, sum[NT];
    m = -INFINITY, l = 0.f;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) sum[t][r] = 0.f;
    // Tile by tile: scores from the fp32 instruction, lane half j with four of eight dimensions, here against the
    // running maximum; the products with V likewise where every row sees the whole tile, else key by key (what a row
    // does not see it does not multiply by zero either).
    const int last = min(kt1 * 32 - 1, w_hi_max);
#pragma clang loop unroll(disable)
    for (int kt = max(kt0, w_lo_min >> 5); kt * 32 <= last; ++kt) {
      const int first = kt * 32;
      const bool whole = first >= w_lo_max && first + 31 <= w_hi_min;
      const unsigned long long key_row = (unsigned)min(first + n, b_hi);
      const float *kp = a.kv + key_row * kv_stride + h * dn, *rp = a.key_rot + key_row * sh.row_w;
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = 0.f;
      auto dot = [&](const float *kd, const float *qd, int dims) {
#pragma clang loop unroll(disable)
        for (int d0 = 0; d0 < dims; d0 += 16) {
          f32x4 kv[2], qv[2];
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const int d = d0 + 8 * u + 4 * j;
            kv[u] = d < dims ? *(const f32x4 *)(kd + d) : f32x4{0.f, 0.f, 0.f, 0.f};
            qv[u] = d < dims ? *(const f32x4 *)(qd + d) * a.c : f32x4{0.f, 0.f, 0.f, 0.f};
          }
#pragma unroll
          for (int i = 0; i < 8; ++i) s = mfma_f32(kv[i >> 2][i & 3], qv[i >> 2][i & 3], s);
        }
      };
      dot(kp, q_row, dn);
      dot(rp, q_row + dn, dr);
      float mx = -INFINITY;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = first + 8 * (r >> 2) + 4 * j + (r & 3);
        if (!whole && (key < my_lo || key > my_hi)) s[r] = -INFINITY;
        mx = fmaxf(mx, s[r]);
      }
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      if (mx > m) {
        const float alpha = m == -INFINITY ? 0.f : fast_exp2(m - mx);
        m = mx;
        l *= alpha;
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r) sum[t][r] *= alpha;
      }
      const float mref = m == -INFINITY ? 0.f : m;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[r] = fast_exp2(s[r] - mref);
        l += s[r];
      }
      if (whole) {
        typedef float vrow_t __attribute__((ext_vector_type(NT)));
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const unsigned long long key = (unsigned)(first + 8 * (r >> 2) + 4 * j + (r & 3));
          const vrow_t v = *(const vrow_t *)(v_src + key * kv_stride + (NT * n < sh.vdim ? NT * n : 0));
#pragma unroll
          for (int t = 0; t < NT; ++t) sum[t] = mfma_f32(v[t], s[r], sum[t]);
        }
        continue;
      }
#pragma clang loop unroll(disable)
      for (int r = 0; r < 16; ++r) {
        const float own = s[0], other = __shfl_xor(own, 32);
#pragma unroll
        for (int i = 0; i < 15; ++i) s[i] = s[i + 1];  // (no register is indexed by a loop counter)
#pragma clang loop unroll(disable)
        for (int half = 0; half < 2; ++half) {
          const int key = first + 8 * (r >> 2) + 4 * half + (r & 3);
          if (key < my_lo || key > my_hi) continue;
          const float e = half == j ? own : other;
          const float *vr = v_src + (unsigned long long)(unsigned)key * kv_stride;
#pragma unroll
          for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int w = 0; w < NT; ++w) {  // floats 4 w .. 4 w + 3 of the 4 NT columns that registers 4 q .. 4 q + 3 hold
              const int d = NT * (8 * q + 4 * j) + 4 * w;
              const f32x4 v = *(const f32x4 *)(vr + (d < sh.vdim ? d : 0));
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const int at = 4 * w + i;
                sum[at % NT][4 * q + at / NT] = fmaf(e, v[i], sum[at % NT][4 * q + at / NT]);
              }
            }
        }
      }
    }
    // (one by one through registers of their own: as whole accumulators the loop above would move them about)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float x = sum[t][r];
        asm volatile("" : "+v"(x));
        o[t][r] = x;
      }
  } else {
#pragma unroll
    for (int t = 0; t < NT; ++t) o[t] *= kDropOne;
  }

  l += __shfl_xor(l, 32);
  if (a.splits > 1) {
    const long long pbase = (((long long)item * sh.H + h) * a.splits + chunk) * 128 + wave * 32 + n;
    float *op = a.part_o + pbase * VSTR;
#pragma unroll
    for (int r = 0; r < 16; ++r)
#pragma unroll
      for (int t = 0; t < NT; t += 2)
        *(float2 *)(op + NT * (8 * (r >> 2) + 4 * j + (r & 3)) + t) = float2{o[t][r], o[t + 1][r]};
    if (j == 0) *(float2 *)(a.part_ml + 2 * pbase) = float2{m, l};
    return;
  }
  if (w_row0 + n >= a.T) return;
  const float sk = a.sink[h] * kLog2e, mf = fmaxf(m, sk);
  const float f = fast_exp2(m - mf), den = l * f + fast_exp2(sk - mf);
  const float factor = f / den * sigmoid1(a.r.raw[(long long)my_row * a.r.stride + a.r.gate_off + h]);
  float *op = a.out + ((long long)my_row * sh.H + h) * sh.vdim;
#pragma unroll
  for (int r = 0; r < 16; ++r)
#pragma unroll
    for (int t = 0; t < NT; t += 2) {
      const int d = NT * (8 * (r >> 2) + 4 * j + (r & 3)) + t;
      if (d < sh.vdim) *(float2 *)(op + d) = float2{o[t][r] * factor, o[t + 1][r] * factor};
    }
}

// Merges the key chunks of one (row block, head), sink and gate included; blockIdx.y: 32 of its rows.
__global__ __launch_bounds__(256) void latent_prefill_combine_kernel(const LatentPrefillArgs a, int vstr) {
  const LatentShape &sh = a.sh;
  const int h = blockIdx.x % sh.H, item = blockIdx.x / sh.H, v4 = sh.vdim >> 2;
  const long long base = ((long long)item * sh.H + h) * a.splits * 128;
  const float sk = a.sink[h] * kLog2e;
  for (int i = threadIdx.x; i < 32 * v4; i += 256) {
    const int rl = blockIdx.y * 32 + i / v4, c = i % v4, row = item * 128 + rl;
    if (row >= a.T) continue;
    float mm = sk;
    for (int s = 0; s < a.splits; ++s) mm = fmaxf(mm, a.part_ml[2 * (base + (long long)s * 128 + rl)]);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    float den = fast_exp2(sk - mm);
    for (int s0 = 0; s0 < a.splits; s0 += 4) {
      f32x4 x[4];
      float2 ml[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const long long p = base + (long long)min(s0 + u, a.splits - 1) * 128 + rl;
        x[u] = *(const f32x4 *)(a.part_o + p * vstr + 4 * c);
        ml[u] = *(const float2 *)(a.part_ml + 2 * p);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (s0 + u >= a.splits) break;
        const float f = fast_exp2(ml[u].x - mm);  // 0 for a chunk in which the row saw no key
        acc += f * x[u];
        den += f * ml[u].y;
      }
    }
    const float g = sigmoid1(a.r.raw[(long long)row * a.r.stride + a.r.gate_off + h]);
    *(f32x4 *)(a.out + ((long long)row * sh.H + h) * sh.vdim + 4 * c) = acc * (g / den);
  }
}

constexpr size_t kMaxLds = 160 * 1024;

bool shape_ok(const LatentShape &sh) {
  return sh.H > 0 && sh.dim > 0 && sh.rot_dim >= 0 && sh.vdim > 0 && sh.kv_rank > 0 && sh.rot_dims >= 0 &&
         sh.rot_dims <= sh.rot_dim && (sh.rot_dims & 1) == 0 && sh.row_w == latent_row_width(sh.kv_rank, sh.rot_dim) &&
         sh.window >= 0;
}
bool rows_ok(const LatentRows &r, const LatentShape &sh, int T) {
  return shape_ok(sh) && T > 0 && r.raw && r.kv_norm && (r.rope_tab || !sh.rot_dims) && r.rows && r.start_pos >= 0 &&
         r.start_row >= 0 && r.kv_off >= 0 && r.gate_off >= 0 && r.stride >= r.kv_off + sh.kv_rank + sh.rot_dim &&
         r.stride >= r.gate_off + sh.H;
}

}  // namespace

hipError_t launch_latent_append(const LatentRows &r, const LatentShape &sh, int T, float *q, hipStream_t stream) {
  if (!rows_ok(r, sh, T)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(latent_append_kernel, dim3((unsigned)T), dim3(256), 0, stream, r, sh, q);
  return hipGetLastError();
}

hipError_t launch_latent_absorb(const float *q, const float *uk, const LatentRows &r, const LatentShape &sh, int T,
                                float *q_abs, hipStream_t stream) {
  if (!rows_ok(r, sh, T) || !q || !uk || !q_abs) return hipErrorInvalidValue;
  const int rt = T == 1 ? 1 : 4;
  const size_t lds = (size_t)rt * (sh.dim + 4 * 64) * sizeof(float);
  const long long wgs = (long long)T + (long long)((sh.kv_rank + 63) / 64) * sh.H * ((T + rt - 1) / rt);
  if (lds > 64 * 1024 || wgs > 0x7fffffffLL) return hipErrorInvalidValue;
  const float qscale = sh.scale * kLog2e;
  if (rt == 1)
    hipLaunchKernelGGL(latent_absorb_kernel<1>, dim3((unsigned)wgs), dim3(256), lds, stream, q, uk, r, sh, T, q_abs, qscale);
  else
    hipLaunchKernelGGL(latent_absorb_kernel<4>, dim3((unsigned)wgs), dim3(256), lds, stream, q, uk, r, sh, T, q_abs, qscale);
  return hipGetLastError();
}

bool plan_latent_absorbed(const LatentShape &sh, int T, int start_row, LatentPlan &p) {
  if (!shape_ok(sh) || T < 1 || start_row < 0 || (long long)T * sh.H > 0x3fffffff) return false;
  p.v_w = (sh.kv_rank + 15) / 16 * 16;
  p.v_slices = (p.v_w + 1023) / 1024;
  // (what fits 160 KiB: rows of up to 800 floats in steps of 32, up to 1200 in steps of 16)
  p.key_tile = sh.row_w <= 800 ? 32 : 16;
  const size_t ldr = (size_t)sh.row_w + 4;
  p.lds_bytes = ((16 + p.key_tile) * ldr + (size_t)8 * 16 * 17) * sizeof(float);
  if (p.lds_bytes > kMaxLds) return false;
  p.col_tiles = (T * sh.H + 15) / 16;
  // the most keys a tile of columns walks: what the last of its rows sees and the rows before it saw besides
  int span = (14 + sh.H) / sh.H + 1;  // rows that 16 consecutive (row, head) pairs can touch
  if (span > T) span = T;
  long long keys = (long long)start_row + T;
  if (sh.window && keys > (long long)sh.window + span - 1) keys = (long long)sh.window + span - 1;
  const int tiles = (int)((keys + p.key_tile - 1) / p.key_tile);
  static const int target_knob = getenv("SHAINET_HIP_LATENT_WGS") ? atoi(getenv("SHAINET_HIP_LATENT_WGS")) : 0;
  const int target = target_knob > 0 ? target_knob : 256;
  int splits = target / p.col_tiles;
  if (splits > 128) splits = 128;
  if (splits > tiles) splits = tiles;
  if (splits < 1) splits = 1;
  p.tiles_per_split = (tiles + splits - 1) / splits;
  p.splits = (tiles + p.tiles_per_split - 1) / p.tiles_per_split;
  p.partial_floats = (size_t)p.col_tiles * 16 * p.splits * (p.v_w + 2);
  return true;
}

hipError_t launch_latent_absorbed(const float *q_abs, const float *rows, float *partials, const LatentShape &sh, int T,
                                  int start_row, const LatentPlan &p, hipStream_t stream) {
  LatentPlan want;
  if (!q_abs || !rows || !partials || !plan_latent_absorbed(sh, T, start_row, want) || want.splits != p.splits ||
      want.partial_floats != p.partial_floats || p.splits > 65535)
    return hipErrorInvalidValue;
  float *part_o = partials, *part_ml = partials + (size_t)p.col_tiles * 16 * p.splits * p.v_w;
  const dim3 grid((unsigned)p.col_tiles, (unsigned)p.splits, (unsigned)p.v_slices);
  const int slice = p.v_w < 1024 ? p.v_w : 1024;
  const int ntw = (slice / 16 + 7) / 8;
#define SHAINET_LAUNCH_ABSORBED(KT_, NTW_)                                                                               \
  do {                                                                                                                   \
    static const hipError_t a_ = hipFuncSetAttribute((const void *)latent_absorbed_kernel<KT_, NTW_>,                           \
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxLds);                 \
    if (a_ != hipSuccess) return a_;                                                                                    \
    hipLaunchKernelGGL((latent_absorbed_kernel<KT_, NTW_>), grid, dim3(512), p.lds_bytes, stream, q_abs, rows, part_o,  \
                       part_ml, sh, T, start_row, p.splits, p.tiles_per_split, p.v_w);                                  \
  } while (0)
#define SHAINET_LAUNCH_ABSORBED_K(NTW_)  \
  do {                                   \
    if (p.key_tile == 32)                \
      SHAINET_LAUNCH_ABSORBED(32, NTW_); \
    else                                 \
      SHAINET_LAUNCH_ABSORBED(16, NTW_); \
  } while (0)
  if (ntw <= 1)
    SHAINET_LAUNCH_ABSORBED_K(1);
  else if (ntw <= 2)
    SHAINET_LAUNCH_ABSORBED_K(2);
  else if (ntw <= 4)
    SHAINET_LAUNCH_ABSORBED_K(4);
  else
    SHAINET_LAUNCH_ABSORBED_K(8);
#undef SHAINET_LAUNCH_ABSORBED_K
#undef SHAINET_LAUNCH_ABSORBED
  return hipGetLastError();
}

hipError_t launch_latent_out(const float *partials, const float *uv, const float *sink, const LatentRows &r,
                             const LatentShape &sh, int T, const LatentPlan &p, float *out, hipStream_t stream) {
  if (!rows_ok(r, sh, T) || !partials || !uv || !sink || !out || sh.H > 65535) return hipErrorInvalidValue;
  const float *part_ml = partials + (size_t)p.col_tiles * 16 * p.splits * p.v_w;
  const int rt = T == 1 ? 1 : 4;
  const int v4 = p.v_w / 4;
  if (v4 > 1024) return hipErrorInvalidValue;
  const size_t lds = ((size_t)rt * (p.v_w + p.splits) + (size_t)(1024 / v4) * p.v_w) * sizeof(float);
  const long long wgs = (long long)((sh.vdim + 15) / 16) * sh.H;
  if (lds > 64 * 1024 || (T + rt - 1) / rt > 65535 || wgs > 0x7fffffffLL) return hipErrorInvalidValue;
  const dim3 grid((unsigned)wgs, (unsigned)((T + rt - 1) / rt));
  if (rt == 1)
    hipLaunchKernelGGL(latent_out_kernel<1>, grid, dim3(1024), lds, stream, partials, part_ml, uv, sink, r, sh, T, p.splits,
                       p.v_w, out);
  else
    hipLaunchKernelGGL(latent_out_kernel<4>, grid, dim3(1024), lds, stream, partials, part_ml, uv, sink, r, sh, T, p.splits,
                       p.v_w, out);
  return hipGetLastError();
}

bool latent_row_fits(const LatentShape &sh, int start_row) {
  // (the times above, less 5.4 us for a launch and its meetings: 0.047 us per 1000 floats of a head's weights, 0.04 of the keys', in rows
  // as wide as the form's lanes take them: 1100 keys of 80 floats 17.6 us, of 144 17.7;  600 keys of 352 22.1, of 416 20.6.  The three launches
  // take 18 us and more, of more than 64 heads 24 and more: a step of a layer, the launches beside these included, three | this, 128
  // heads of 64 + 32 and 64, latents of 256, 800 keys 44.7 | 38.0, 1100 47.4 | 43.9;  of 128 + 64 and 128, latents of 512, 480 keys 73 | 60)
  const long long keys = sh.window && start_row >= sh.window ? sh.window : (long long)start_row + 1, row = sh.row_w <= 320 ? 288 : 576;
  return shape_ok(sh) && start_row >= 0 && (sh.kv_rank & 3) == 0 && sh.row_w <= 576 && sh.H <= 256 &&
         47LL * (sh.dim + sh.vdim) * (row == 288 ? 256 : 512) + 40 * keys * row <= (sh.H <= 64 ? 12600000 : row == 288 ? 17600000 : 19000000);
}

hipError_t launch_latent_row(const float *q, const float *uk, const float *uv, const float *sink, const LatentRows &r,
                             const LatentShape &sh, float *out, hipStream_t stream) {
  if (!rows_ok(r, sh, 1) || !latent_row_fits(sh, r.start_row) || !q || !uk || !uv || !sink || !out ||
      (((uintptr_t)uk | (uintptr_t)uv | (uintptr_t)r.rows) & 15))
    return hipErrorInvalidValue;
  const float qscale = sh.scale * kLog2e;
#define SHAINET_LAUNCH_LATENT_ROW(P_, G_, RK_, RV_)                                                                          \
  hipLaunchKernelGGL((latent_row_kernel<P_, G_, RK_, RV_>), dim3((unsigned)sh.H), dim3(512), 0, stream, q, uk, uv, sink, r, sh, qscale, out)
  if (sh.row_w <= 320)
    SHAINET_LAUNCH_LATENT_ROW(5, 4, 2, 2);
  else
    SHAINET_LAUNCH_LATENT_ROW(9, 2, 2, 1);
#undef SHAINET_LAUNCH_LATENT_ROW
  return hipGetLastError();
}

bool plan_latent_expanded(const LatentShape &sh, int T, int start_row, LatentExpandedPlan &p) {
  if (!shape_ok(sh) || T < 1 || start_row < 0) return false;
  // 16-byte pieces of the query, key and value rows
  if ((sh.dim | sh.rot_dim | sh.vdim | sh.kv_rank) & 3) return false;
  const int dk = (sh.dim + 7) / 8 * 8 + (sh.rot_dim + 7) / 8 * 8;
  if (dk > 256 || sh.vdim > 128) return false;
  p.nk = dk <= 96 ? 12 : dk <= 128 ? 16 : dk <= 192 ? 24 : 32;
  p.nt = sh.vdim <= 64 ? 2 : 4;
  const int back = sh.window && sh.window - 1 < start_row ? sh.window - 1 : start_row;
  p.first_row = start_row - back;
  p.key_rows = back + T;
  p.items = (T + 127) / 128;
  const long long blocks = (long long)p.items * sh.H;
  if (blocks > 0x3fffff) return false;
  int tiles = (p.key_rows + 31) / 32;  // of the row block with the most keys
  if (sh.window && tiles > (sh.window + 127) / 32 + 2) tiles = (sh.window + 127) / 32 + 2;
  static const int splits_knob = getenv("SHAINET_HIP_LATENT_SPLITS") ? atoi(getenv("SHAINET_HIP_LATENT_SPLITS")) : 0;
  int splits = blocks >= 384 ? 1 : (int)((512 + blocks - 1) / blocks);  // two workgroups per compute unit
  if (splits > tiles / 4) splits = tiles / 4;
  if (splits > 16) splits = 16;
  if (splits_knob > 0) splits = splits_knob;
  p.splits = splits < 1 ? 1 : splits;
  p.partial_floats = p.splits > 1 ? (size_t)blocks * p.splits * 128 * (p.nt * 32 + 2) : 0;
  // Multiply-adds: per (row, key, head) this form's and the absorbed form's, whose kernel reaches about half
  // this one's rate; and the products, here of every key row and at twice the rate (the library's), there of the new
  // rows alone.  A few rows behind many keys are the absorbed form's, whose tiles of columns hold 32 rows (16 heads) as
  // cheaply as 17.  A pass of three layers, 16 heads of 96 and 64 | 192 and 128 dimensions, us, absorbed : expanded:
  //   keys in front   17 rows               32 rows               36 rows               48 rows
  //        40      387:364 | 605:582     410:371 | 664:602     470:395 | 738:645     474:401 | 785:657
  //       100      402:389 | 612:620     433:399 | 676:644     474:417 | 747:689     479:423 | 794:691
  //       200      412:415 | 620:664     436:419 | 677:658     491:433 | 758:697     505:446 | 794:704
  //       500      430:478 | 635:724     461:480 | 706:738     509:494 | 775:778     519:496 | 826:777
  //      3000      426:510 | 784:964     488:508 | 893:982     530:526 | 1027:1030   560:530 | 1172:1040
  const double pairs = (double)T * (sh.window && sh.window < p.key_rows ? sh.window : p.key_rows);
  const double product = (double)sh.kv_rank * sh.H * (sh.dim + sh.vdim);
  const double here = pairs * sh.H * (8 * p.nk + 32 * p.nt) + 0.5 * p.key_rows * product;
  const double there = 2.0 * pairs * sh.H * (sh.row_w + sh.kv_rank) + T * product;
  p.pays = T > 16 && (T > 32 || p.key_rows <= 160) && here < there;
  return true;
}

hipError_t launch_latent_expanded(const float *q, const float *kv, const float *sink, const LatentRows &r,
                                  const LatentShape &sh, int T, const LatentExpandedPlan &p, float *partials, float *out,
                                  hipStream_t stream) {
  LatentExpandedPlan want;
  if (!rows_ok(r, sh, T) || !q || !kv || !sink || !out || !plan_latent_expanded(sh, T, r.start_row, want) ||
      want.splits != p.splits || want.key_rows != p.key_rows || (p.splits > 1 && !partials))
    return hipErrorInvalidValue;
  if (((uintptr_t)q | (uintptr_t)kv | (uintptr_t)r.rows | (uintptr_t)out | (uintptr_t)partials) & 15) return hipErrorInvalidValue;
  LatentPrefillArgs a = {};
  a.q = q;
  a.kv = kv;
  a.key_rot = r.rows + (long long)p.first_row * sh.row_w + sh.kv_rank;
  a.sink = sink;
  a.r = r;
  a.sh = sh;
  a.out = out;
  a.part_o = partials;
  a.part_ml = partials ? partials + (size_t)p.items * sh.H * p.splits * 128 * p.nt * 32 : nullptr;
  a.T = T;
  a.first_key = r.start_row - p.first_row;
  a.items = p.items;
  a.splits = p.splits;
  a.c = sh.scale * kLog2e;
  const dim3 grid((unsigned)(p.items * sh.H * p.splits));
#define SHAINET_LAUNCH_EXPANDED(NK_)                                                               \
  do {                                                                                             \
    if (p.nt == 2)                                                                                 \
      hipLaunchKernelGGL((latent_prefill_kernel<NK_, 2>), grid, dim3(256), 0, stream, a);          \
    else                                                                                           \
      hipLaunchKernelGGL((latent_prefill_kernel<NK_, 4>), grid, dim3(256), 0, stream, a);          \
  } while (0)
  switch (p.nk) {
    case 12: SHAINET_LAUNCH_EXPANDED(12); break;
    case 16: SHAINET_LAUNCH_EXPANDED(16); break;
    case 24: SHAINET_LAUNCH_EXPANDED(24); break;
    default: SHAINET_LAUNCH_EXPANDED(32); break;
  }
#undef SHAINET_LAUNCH_EXPANDED
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || p.splits == 1) return e;
  hipLaunchKernelGGL(latent_prefill_combine_kernel, dim3((unsigned)(p.items * sh.H), 4), dim3(256), 0, stream, a, p.nt * 32);
  return hipGetLastError();
}

}  // namespace shainet
