// Causal grouped-query attention over the device KV cache for gfx950 (CDNA4).
//
// Together with decode_kernel.hip (one new row per sequence) these kernels replace
// attention_heads_cpu (llama_block.cr:302-401) and the reference's
// attention_kv_kernel (cuda_kernels.cu:734-806):
//
//   prefill_mfma_kernel   many new rows.  Query rows and the heads of a group
//       are flattened into "virtual rows"; a wavefront owns 32 of them, a
//       workgroup 128.  K/V tiles of 32 keys are split into bf16 parts on their way
//       to LDS and consumed by v_mfma_f32_32x32x16_bf16.
//   generic_attn_kernel   any head_dim; one wavefront per (row, head).  Used for
//       head dims other than 64 and 128.
//
// The MFMA kernels compute S^T = K Q^T so that the probabilities come out of the MFMA
// accumulator already laid out as the B operand of O^T = V^T P^T: no transpose,
// no LDS round trip for P.  The contraction index of an MFMA may be visited in
// any order as long as A and B agree.
#include "attn_kernels.hpp"
#include "split_mfma.hpp"

#include <math.h>
#include <stdlib.h>
#include <string.h>

namespace shainet {

namespace {

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

__device__ __forceinline__ int find_seq(const SeqTable &st, int item, const int *off) {
  int s = 0;
  while (s + 1 < st.n_seqs && item >= off[s + 1]) ++s;
  return s;
}

// ---------------------------------------------------------------------------
// Prefill: MFMA 32x32x16, K/V tiles staged through LDS.
//
// Virtual row v of a (sequence, kv head): query row v / g, head kvh*g + v % g.
// MFMA layout (lane l, j = l/32): A[m = l%32][k = 8j .. 8j+7], B[k = 8j .. 8j+7][n = l%32],
// D[m = 8*(r/4) + 4*j + r%4][n = l%32] for accumulator register r = 0..15.
//   scores:  m = key within the tile, n = virtual row, k = d.
//   output:  tile t, m = d index (d = NT*m + t), contraction over the tile's keys in
//            the order the score accumulator holds them.
// Row block number `rank` in dispatch order -> (sequence, block).  Level 0 is every
// sequence's last block (the longest key range), level 1 the one before, and so
// on.  st.work_off[s] = row blocks of sequence s, st.ord = sequences by descending
// block count.
__device__ __forceinline__ void locate_block(const SeqTable &st, int rank, int &s, int &vb) {
  s = 0;
  int level = 0;
  for (int b = st.n_seqs - 1; b >= 0; --b) {  // levels [n_{b+1}, n_b) have b+1 active sequences
    const int lo = b + 1 < st.n_seqs ? st.work_off[st.ord[b + 1]] : 0;
    const int cnt = (st.work_off[st.ord[b]] - lo) * (b + 1);
    if (rank < cnt) {
      level = lo + rank / (b + 1);
      s = st.ord[rank % (b + 1)];
      break;
    }
    rank -= cnt;
  }
  vb = st.work_off[s] - 1 - level;
}

// Units of 16 bytes (eight bf16, one MFMA operand of a lane) that one key tile takes in LDS.  K: [part][octet of
// d][key], an octet's 32 keys one unit apart from a multiple of 16 (a row's octets are written side by side).  V:
// [part][group of eight keys][column], column d at place d / NT of block d % NT, four units of padding a block; group
// 2 u + j holds the keys 16 u + 4 j + {0 .. 3, 8 .. 11}, the ones whose probabilities lane half j has in its
// registers 8 u .. 8 u + 7.
template <int HD>
struct TileUnits {
  static constexpr int NT = HD / 32;
  static constexpr int kOctK = 33, kPartK = HD / 8 * kOctK;
  static constexpr int kGroupV = NT * 36, kPartV = 4 * kGroupV;
  static constexpr int kK = 3 * kPartK, kTile = kK + 3 * kPartV;
};

// G = 1: four wavefronts, each with 32 virtual rows, walk the key tiles together.
// G = 2: eight wavefronts; wavefronts 4..7 own the same rows as 0..3 and take every
// second key tile, so that each SIMD holds two wavefronts of one workgroup and the
// waits and vector instructions of one hide behind the MFMAs of the other
// even when a launch puts a single workgroup on a compute unit.  The two
// halves merge through LDS.
// One workgroup's work: the row block (and key chunk) number `bid` of the launch.
// PAD: the head dimension of the data (sh.hd, a multiple of 4) is smaller than HD, the one the
// tiles are laid out for: query elements beyond it are zeros (whatever stands in for the keys'
// there does not reach the scores), output elements beyond it are not stored, and a tile's
// pieces beyond it repeat the row's first piece (a cache hit, no HBM traffic).
// BIAS (with PAD): scores gain a value by distance (DistanceBias), value rows have a width of their own.
//
// Queries, keys, values and probabilities enter the MFMAs as exact sums of three bf16 numbers
// (split_mfma.hpp): the queries once, a key tile by the workgroup on its way to LDS, the probabilities in
// the registers the scores came in.  A tile costs a wavefront HD / 16 x 6 + HD / 16 x 6 MFMAs of 32 cycles (64:
// 1536) where the fp32 instruction took HD x 64 (4096), and about as many cycles of vector instructions, which run
// beside them.  Kernel times, the fp32 instruction before (us): 2048 rows, 32 / 8 heads of 64, 99 (146), 8192 rows 1324
// (2050); 512 rows on 16384 cached, 32 / 4 heads of 128, 684 (1056); 2048 rows, 32 / 8 heads of 128, 186 (279).
// Bound by the power the card may draw, as the large products are; raising one group's priority changes nothing and
// parking V between the score MFMAs costs 5 to 16 %.  (Queries and keys as two fp16 numbers and scores of three products
// took 14 and 17 % less, but such numbers leave out up to 2^-21 of a product, and where a key's second parts have the signs of the
// query's that adds up.)
template <int HD, bool SPLIT, int G, bool PAD, bool BIAS>
__device__ __forceinline__ void prefill_block(const int bid, const float *__restrict__ q_rot,
                                              const float *__restrict__ kc, const float *__restrict__ vc,
                                              float *__restrict__ out, float *__restrict__ part_o,
                                              float *__restrict__ part_ml, const SeqTable &st, const Shape &sh,
                                              int ns, float c, const DistanceBias &db) {
  static_assert(PAD || !BIAS, "sizes of their own come with padding");
  using U = TileUnits<HD>;
  constexpr int KS = HD / 16;   // MFMA steps along d of the scores
  constexpr int NT = HD / 32;   // d tiles of the output
  constexpr int NI = HD / 64;   // items per thread to stage the G K (or V) tiles of one step
  constexpr int NTHREADS = 256 * G;
  __shared__ __attribute__((aligned(16))) u32x4 lds[G * U::kTile];

  // Workgroups are numbered so that the hardware dispatcher, which hands them out in
  // index order, starts the row blocks with the longest key ranges first; the kv
  // head is the fastest index, so with 8 kv heads each XCD (index % 8) keeps to one
  // head and its K/V stay in that XCD's L2.  When a launch has too few row blocks to
  // fill the chip, each block's key range is cut into ns chunks that run as separate
  // workgroups and leave partial (max, sum, O) rows for prefill_combine_kernel.
  const int kvh = bid % sh.KV;
  const int chunk = SPLIT ? (bid / sh.KV) % ns : 0;
  const int item = SPLIT ? bid / sh.KV / ns : bid / sh.KV;
  int s, vb;
  locate_block(st, item, s, vb);
  // These are the same for all lanes of a wavefront, which the compiler cannot see: said so,
  // tile counts, loop conditions and address bases live in scalar registers
  auto uniform = [](int x) { return __builtin_amdgcn_readfirstlane(x); };
  s = uniform(s);
  vb = uniform(vb);
  const int g = sh.g, T = st.n_new[s], S = st.start_pos[s];
  const int L = S + T, VR = T * g;
  const int lane = threadIdx.x & 63;
  const int wave = uniform((threadIdx.x >> 6) & 3);  // which 32 virtual rows of the block
  const int gidx = uniform(threadIdx.x >> 8);        // which share of the key tiles (always 0 for G = 1)
  const int n = lane & 31, j = lane >> 5;
  const int v0 = vb * 128 + wave * 32;
  const bool wave_active = v0 < VR;
  const int my_v = v0 + n;
  const bool valid = my_v < VR;
  const int row = valid ? my_v / g : T - 1;
  const int hg = valid ? my_v - row * g : 0;
  const int lim = S + row;                                            // last visible key of this lane's row
  const int wave_lo = S + (wave_active ? v0 / g : 0);                 // smallest lim in the wavefront
  const int wave_hi = wave_active ? S + min(v0 + 31, VR - 1) / g : -1;  // largest
  const int wg_hi = S + min(vb * 128 + 127, VR - 1) / g;
  const int n_tiles = wg_hi / 32 + 1;
  const int tiles_per_chunk = SPLIT ? (n_tiles + ns - 1) / ns : n_tiles;
  const int kt0 = chunk * tiles_per_chunk, kt1 = min(n_tiles, kt0 + tiles_per_chunk);
  const int hd = PAD ? uniform(sh.hd) : HD;  // floats between two rows of q, K, V and the output
  const long long head_base = (long long)st.slot[s] * sh.seq_stride + (long long)kvh * sh.cap * hd;
  const float *kbase = kc + head_base;
  const int vhd = BIAS ? uniform(db.v_hd) : hd;
  const float *vbase = vc + (BIAS ? ((long long)st.slot[s] * sh.KV + kvh) * sh.cap * vhd : head_base);
  const long long qo_off = ((long long)(st.tok_off[s] + row) * sh.H + kvh * g + hg) * vhd;  // of the row's result
  const long long q_off = BIAS ? (st.tok_off[s] + row) * db.q_stride + (long long)(kvh * g + hg) * hd : qo_off;
  // entry of key row k: bias_row[k]
  const float *bias_row = BIAS ? db.tab + (long long)(kvh * g + hg) * db.stride + (db.origin - lim) : nullptr;

  // what a thread stages of a step's G tiles: K, an octet of d of a row; V, eight rows of a column
  unsigned k_off[NI], v_off[NI];
  int k_row[NI], v_row[NI], k_unit[NI], v_unit[NI];
  bool k_second[NI];  // the octet's second half lies within the row
#pragma unroll
  for (int u = 0; u < NI; ++u) {
    const int idx = threadIdx.x + NTHREADS * u;
    const int oct = idx % (HD / 8), r = idx / (HD / 8);
    k_row[u] = r;
    k_off[u] = PAD && 8 * oct >= hd ? 0u : 32u * oct;
    k_second[u] = !PAD || 8 * oct + 4 < hd;
    k_unit[u] = (r >> 5) * U::kTile + oct * U::kOctK + (r & 31);
    const int d = idx % HD, group = idx / HD & 3, ts = idx / (4 * HD);
    v_row[u] = 32 * ts + 16 * (group >> 1) + 4 * (group & 1);
    v_off[u] = PAD && d >= vhd ? 0u : 4u * d;
    v_unit[u] = ts * U::kTile + U::kK + group * U::kGroupV + d % NT * 36 + d / NT;
  }
  const unsigned k_stride = (unsigned)hd * 4, v_stride = (unsigned)vhd * 4;
  f32x4 stage_k[NI][2];
  float stage_v[NI][8];
  // a scalar base and a 32-bit byte offset per lane (a head's rows span less than 4 GiB: checked
  // at launch); rows past the last one repeat it
  auto load_k = [&](int sp) {
    const int first = (kt0 + G * sp) * 32;
#pragma unroll
    for (int u = 0; u < NI; ++u) {
      const char *p = (const char *)kbase + ((unsigned)min(first + k_row[u], L - 1) * k_stride + k_off[u]);
      stage_k[u][0] = *(const f32x4 *)p;
      stage_k[u][1] = *(const f32x4 *)(p + (k_second[u] ? 16 : 0));
    }
  };
  auto load_v = [&](int sp) {
    const int first = (kt0 + G * sp) * 32;
    if (first + 32 * G <= L) {
      const char *base = (const char *)vbase + (unsigned long long)first * v_stride;
#pragma unroll
      for (int u = 0; u < NI; ++u) {
        const unsigned off = (unsigned)v_row[u] * v_stride + v_off[u];
#pragma unroll
        for (int i = 0; i < 8; ++i) stage_v[u][i] = *(const float *)(base + (unsigned long long)((i & 3) + 8 * (i >> 2)) * v_stride + off);
      }
    } else {
#pragma unroll
      for (int u = 0; u < NI; ++u)
#pragma unroll
        for (int i = 0; i < 8; ++i)
          stage_v[u][i] = *(const float *)((const char *)vbase +
                                           ((unsigned)min(first + v_row[u] + (i & 3) + 8 * (i >> 2), L - 1) * v_stride + v_off[u]));
    }
  };
  auto park_k = [&]() {
#pragma unroll
    for (int u = 0; u < NI; ++u) {
      u32x4 h, m, l;
      split_octet(stage_k[u][0], stage_k[u][1], h, m, l);
      lds[k_unit[u]] = h;
      lds[k_unit[u] + U::kPartK] = m;
      lds[k_unit[u] + 2 * U::kPartK] = l;
    }
  };
  auto park_v = [&]() {
#pragma unroll
    for (int u = 0; u < NI; ++u) {
      u32x4 h, m, l;
      split_octet(f32x4{stage_v[u][0], stage_v[u][1], stage_v[u][2], stage_v[u][3]},
                  f32x4{stage_v[u][4], stage_v[u][5], stage_v[u][6], stage_v[u][7]}, h, m, l);
      lds[v_unit[u]] = h;
      lds[v_unit[u] + U::kPartV] = m;
      lds[v_unit[u] + 2 * U::kPartV] = l;
    }
  };

  // steps of G tiles, one per group of wavefronts; below "tile sp" is this group's tile of step sp
  const int n_sp = kt0 < kt1 ? (kt1 - kt0 + G - 1) / G : 0;
  if (n_sp > 0) {
    load_k(0);
    load_v(0);
  }
  // the row's query, scaled by scale * log2(e): scores come out in log2 units
  u32x4 qf[KS][3];
  bool apart;  // some query of the wavefront needs its scores in fp32
  {
    f32x4 t[KS][2];
    const float *qp = q_rot + q_off + 8 * j;
#pragma unroll
    for (int i = 0; i < KS; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        // (lanes past the last virtual row repeat the last row: their results are never used)
        t[i][h] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (!PAD || 16 * i + 8 * j + 4 * h < hd) t[i][h] = *(const f32x4 *)(qp + 16 * i + 4 * h);
      }
#pragma unroll
    for (int i = 0; i < KS; ++i) split_octet(t[i][0] * c, t[i][1] * c, qf[i][0], qf[i][1], qf[i][2]);
    float least = INFINITY, most = 0.f;
#pragma unroll
    for (int i = 0; i < KS; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (PAD && 16 * i + 8 * j + 4 * h >= hd) continue;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const float size = fabsf(t[i][h][w] * c);
          least = fminf(least, size);
          most = fmaxf(most, size);
        }
      }
    apart = false;
    // (looked at closely only where there is a zero or something out of the ordinary)
    if (__builtin_expect(__any(!(least >= 0x1p-109f) || !(most < 0x1p100f)), 0)) {
      QueryRange range;
#pragma clang loop unroll(disable)
      for (int d = 4 * j; d < hd; d += 8) range.add(*(const f32x4 *)(q_rot + q_off + d));
      apart = __any(range.apart(c));
    }
  }

  // Online softmax against a reference value per virtual row instead of the running maximum: m_ref is only moved
  // (and l, O rescaled) when a score exceeds it by more than kTau, or for a row's first visible key;
  // probabilities are then at most 2^kTau, no overflow.  A tile on the common path costs a maximum, 16
  // subtractions, exp2 and adds per lane.
  constexpr float kTau = 8.f;
  float m_ref = 0.f, l = 0.f;
  float thr = -INFINITY;  // a row's scores move m_ref when above this: anything finite until its first key, m_ref + kTau after
  f32x16 o[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[t][r] = 0.f;

  // One stage of LDS for K and one for V.  Step sp: scores and softmax of tile sp from K(sp), V(sp) is parked
  // meanwhile; a barrier; O^T += V^T(sp) P^T(sp), K(sp + 1) is parked meanwhile; a barrier.  What is parked was
  // requested a step before.
  const u32x4 *tile = lds + gidx * U::kTile;
  if (n_sp > 0) {
    park_k();
    if (n_sp > 1) load_k(1);
  }
  __syncthreads();
  for (int sp = 0; sp < n_sp; ++sp) {
    const int kt = kt0 + G * sp + gidx;  // this group's tile
    const bool have = kt < kt1 && kt * 32 <= wave_hi;
    // the tile's values by distance are asked for in front of its MFMAs; a tile that lies
    // `reach` or more behind all rows of the wavefront has none
    f32x4 near_bias[BIAS ? 4 : 1];
    const bool near = BIAS && have && wave_lo - (kt * 32 + 31) < db.reach;
    if constexpr (BIAS) {
      if (near) {
        struct __attribute__((packed, aligned(4))) Four { f32x4 v; };
#pragma unroll
        for (int r = 0; r < 4; ++r) near_bias[r] = ((const Four *)(bias_row + kt * 32 + 8 * r + 4 * j))->v;
      }
    }
    f32x16 p;
    if (have) {
      // S^T of the key tile: 32 keys x 32 virtual rows
#pragma unroll
      for (int r = 0; r < 16; ++r) p[r] = 0.f;
      const u32x4 *kl = tile + j * U::kOctK + n;
#pragma unroll
      for (int i = 0; i < KS; ++i) {
        u32x4 kf[3];
#pragma unroll
        for (int w = 0; w < 3; ++w) kf[w] = kl[w * U::kPartK + 2 * i * U::kOctK];
#pragma unroll
        for (int w = 0; w < 6; ++w) p = mfma_bf16(kf[kPartA[w]], qf[i][kPartB[w]], p);
      }
    }
    park_v();
    if (sp + 1 < n_sp) load_v(sp + 1);
    if (have) {
      if constexpr (BIAS) {
        if (near) {
#pragma unroll
          for (int r = 0; r < 16; ++r) p[r] += near_bias[r >> 2][r & 3];
        }
      }
      if (kt * 32 + 31 > wave_lo) {  // tile crosses the diagonal for some row of this wavefront
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = kt * 32 + 8 * (r >> 2) + 4 * j + (r & 3);
          if (key > lim) p[r] = -INFINITY;
        }
      }
      float mx = fmaxf(fmaxf(p[0], p[1]), p[2]);
#pragma unroll
      for (int r = 3; r < 15; r += 2) mx = fmaxf(fmaxf(mx, p[r]), p[r + 1]);
      mx = fmaxf(mx, p[15]);
      // mx covers this lane's half of the row's keys in the tile; the row's maximum is above thr
      // exactly when one of the two halves' is (never for a row without a visible key here:
      // -inf), so the halves only exchange their maxima once a move is certain
      if (__builtin_amdgcn_ballot_w64(mx > thr) != 0) {
        // rare after a row's first tiles: move the reference to this tile's maximum
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        if (mx > thr) {
          const float alpha = thr != -INFINITY ? fast_exp2(m_ref - mx) : 1.f;  // nothing to rescale before a row's first key
          m_ref = mx;
          thr = mx + kTau;
          l *= alpha;
#pragma unroll
          for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[t][r] *= alpha;
        }
      }
      float psum = 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        p[r] = fast_exp2(p[r] - m_ref);
        psum += p[r];
      }
      l += psum;
    }
    __syncthreads();  // V(sp) is there, nobody reads K(sp) any more
    if (have) {
      // O^T += V^T P^T; the probabilities are where the scores were
      const u32x4 *vl = tile + U::kK + j * U::kGroupV + n;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        u32x4 pf[3];
        split_octet(f32x4{p[8 * u], p[8 * u + 1], p[8 * u + 2], p[8 * u + 3]},
                    f32x4{p[8 * u + 4], p[8 * u + 5], p[8 * u + 6], p[8 * u + 7]}, pf[0], pf[1], pf[2]);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          u32x4 vf[3];
#pragma unroll
          for (int w = 0; w < 3; ++w) vf[w] = vl[w * U::kPartV + 2 * u * U::kGroupV + 36 * t];
#pragma unroll
          for (int w = 0; w < 6; ++w) o[t] = mfma_bf16(vf[kPartA[w]], pf[kPartB[w]], o[t]);
        }
      }
    }
    if (sp + 1 < n_sp) park_k();
    if (sp + 2 < n_sp) load_k(sp + 2);
    __syncthreads();  // K(sp + 1) is there, nobody reads V(sp) any more
  }

  // Some results are taken again, tile by tile in fp32:
  //   results that are not finite come from operands that are not, and fp32 says which (8192 rows, 32 / 8 heads of 64, NaN
  //   in key 5: 4.6 ms a call against 1.6 without; key by key, one dimension at a time, it was 279);
  //   queries that ask for it (QueryRange);
  //   values below 2^-110: what they lose by the split, 2^-134 of a key's weight, shows in sums that are themselves small
  //   (the largest weight of a row is 1 or more, all together under 2^30).  Those may be sums of zeros, too: the
  //   values are looked at.  Lifted there by 2^24, or sums of subnormal numbers would round to 2^-149.
  // All values lifted on their way to LDS, and every query looked at closely, cost 8192 rows 5 % (1323 -> 1383 us; this
  // way 1320) and 2048 rows of 32 / 8 heads of 128 4 % (216 -> 224; 218).
  {
    auto size = [](float x) { return __builtin_bit_cast(unsigned, x) << 1; };  // (in the order of |x|)
    float probe = l * 0.f, least = INFINITY;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        probe = fmaf(o[t][r], 0.f, probe);
        least = fminf(least, fabsf(o[t][r]));
      }
    bool again = apart || __any(probe != 0.f);
    float up = 1.f, down = 1.f;
    if (__builtin_expect(__any(least < 0x1p-80f && thr != -INFINITY), 0) && !again) {
      int tid = threadIdx.x;
      asm volatile("" : "+v"(tid));
      unsigned small = ~0u;  // (zeros lie above all)
#pragma clang loop unroll(disable)
      for (int kt = kt0 + gidx; kt < kt1 && kt * 32 <= wave_hi; kt += G) {
        const float *vr = vbase + (long long)min(kt * 32 + (tid & 31), wave_hi) * vhd;
#pragma clang loop unroll_count(4)
        for (int d = (tid & 32) >> 3; d < vhd; d += 8) {
          const f32x4 v = *(const f32x4 *)(vr + d);
#pragma unroll
          for (int i = 0; i < 4; ++i) small = min(small, size(v[i]) - 1u);
        }
      }
      again = __any(small < size(0x1p-109f));
      up = kLift, down = kDropOne;
    }
    if (__builtin_expect(again, 0)) {
      // (what a lane works on is found again from its number: kept for here it would cost the loop above registers)
      int tid = threadIdx.x;
      asm volatile("" : "+v"(tid));
      const int n = tid & 31, j = (tid & 63) >> 5, my_v = min(v0 + n, VR - 1), row = my_v / g, hg = my_v - row * g, lim = S + row;
      const long long q_at = BIAS ? (st.tok_off[s] + row) * db.q_stride + (long long)(kvh * g + hg) * hd
                                  : ((long long)(st.tok_off[s] + row) * sh.H + kvh * g + hg) * hd;
      const float *bias_row = BIAS ? db.tab + (long long)(kvh * g + hg) * db.stride + (db.origin - lim) : nullptr;
      m_ref = 0.f, l = 0.f, thr = -INFINITY;
      f32x16 sum[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) sum[t][r] = 0.f;
      // Tile by tile: scores from the fp32 instruction, lane half j with d = 8 i + 4 j .. + 3 of step i, here against
      // the running maximum; the products with V likewise where every row sees the whole tile, else key by key
      // (what a row does not see it does not multiply by zero either).
#pragma clang loop unroll(disable)
      for (int kt = kt0 + gidx; kt < kt1 && kt * 32 <= wave_hi; kt += G) {
        const int first = kt * 32;
        const bool whole = first + 31 <= wave_lo;
        const float *kr = kbase + (long long)min(first + n, L - 1) * hd + 4 * j, *qr = q_rot + q_at + 4 * j;
        f32x16 p;
#pragma unroll
        for (int r = 0; r < 16; ++r) p[r] = 0.f;
#pragma clang loop unroll(disable)
        for (int d0 = 0; d0 < hd; d0 += 16) {
          f32x4 kv[2], qv[2];
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const int d = d0 + 8 * u;
            const bool in = !PAD || d + 4 * j < hd;
            kv[u] = in ? *(const f32x4 *)(kr + d) : f32x4{0.f, 0.f, 0.f, 0.f};
            qv[u] = in ? *(const f32x4 *)(qr + d) * c : f32x4{0.f, 0.f, 0.f, 0.f};
          }
#pragma unroll
          for (int i = 0; i < 8; ++i) p = mfma_f32(kv[i >> 2][i & 3], qv[i >> 2][i & 3], p);
        }
        if (BIAS && wave_lo - (first + 31) < db.reach) {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int key = first + 8 * (r >> 2) + 4 * j + (r & 3);
            if (key <= lim && lim - key < db.reach) p[r] += bias_row[key];
          }
        }
        float mx = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          if (!whole && first + 8 * (r >> 2) + 4 * j + (r & 3) > lim) p[r] = -INFINITY;
          mx = fmaxf(mx, p[r]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        if (mx > thr) {
          const float alpha = thr == -INFINITY ? 0.f : fast_exp2(thr - mx);
          m_ref = thr = mx;
          l *= alpha;
#pragma unroll
          for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) sum[t][r] *= alpha;
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          p[r] = fast_exp2(p[r] - m_ref);
          l += p[r];
        }
        if (whole) {
          typedef float vrow_t __attribute__((ext_vector_type(NT)));
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int key = first + 8 * (r >> 2) + 4 * j + (r & 3);
            const vrow_t v = *(const vrow_t *)(vbase + (long long)key * vhd + (PAD && NT * n >= vhd ? 0 : NT * n));
#pragma unroll
            for (int t = 0; t < NT; ++t) sum[t] = mfma_f32(v[t] * up, p[r], sum[t]);
          }
          continue;
        }
#pragma clang loop unroll(disable)
        for (int r = 0; r < 16; ++r) {
          const float own = p[0], other = __shfl_xor(own, 32);
#pragma unroll
          for (int i = 0; i < 15; ++i) p[i] = p[i + 1];  // (no register is indexed by a loop counter)
#pragma clang loop unroll(disable)
          for (int h = 0; h < 2; ++h) {
            const int key = first + 8 * (r >> 2) + 4 * h + (r & 3);
            if (key > lim) continue;
            const float e = h == j ? own : other;
            const float *vr = vbase + (long long)key * vhd;
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
              for (int w = 0; w < NT; ++w) {  // floats 4 w .. 4 w + 3 of the 4 NT columns that registers 4 q .. 4 q + 3 hold
                const int d = NT * (8 * q + 4 * j) + 4 * w;
                const f32x4 v = *(const f32x4 *)(vr + (PAD && d >= vhd ? 0 : d));
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                  const int at = 4 * w + i;
                  sum[at % NT][4 * q + at / NT] = fmaf(e, v[i] * up, sum[at % NT][4 * q + at / NT]);
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
          float x = sum[t][r] * down;
          asm volatile("" : "+v"(x));
          o[t][r] = x;
        }
    }
  }

  l += __shfl_xor(l, 32);
  // what the merges below call the maximum: the reference the sums are relative to, in log2
  // units, or -inf for a row that saw no key (its l and O are 0)
  float m = thr == -INFINITY ? -INFINITY : m_ref;
  if constexpr (G == 2) {
    // the second group hands its (max, sum, O) to the first through the tile stages
    // (every wavefront is past the last step's barrier: nobody reads tiles any more)
    float *xo = (float *)lds;                   // [4 row chunks][16 * NT registers][64 lanes]
    float *xm = (float *)lds + 4 * 16 * NT * 64;  // [4][64] max, then [4][64] sum
    static_assert(sizeof lds >= (4 * 16 * NT * 64 + 512) * sizeof(float), "the merge fits the tiles");
    if (gidx == 1) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) xo[((wave * NT + t) * 16 + r) * 64 + lane] = o[t][r];
      xm[wave * 64 + lane] = m;
      xm[256 + wave * 64 + lane] = l;
    }
    __syncthreads();
    if (gidx == 1) return;
    const float m1 = xm[wave * 64 + lane], l1 = xm[256 + wave * 64 + lane];
    const float mnew = fmaxf(m, m1);
    // a side that saw no visible key has max -inf: its factor is 0 (and both may be, in a key chunk)
    const float a0 = m == -INFINITY ? 0.f : fast_exp2(m - mnew);
    const float a1 = m1 == -INFINITY ? 0.f : fast_exp2(m1 - mnew);
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[t][r] = o[t][r] * a0 + xo[((wave * NT + t) * 16 + r) * 64 + lane] * a1;
    l = l * a0 + l1 * a1;
    m = mnew;
  }
  if (SPLIT) {  // unnormalised partial of this key chunk: [128 virtual rows][HD], (max, sum) per row
    const long long pbase = (((long long)item * sh.KV + kvh) * ns + chunk) * 128 + wave * 32 + n;
    float *op = part_o + pbase * HD;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int d = NT * (8 * (r >> 2) + 4 * j + (r & 3));
      if constexpr (NT == 2) {
        *(float2 *)(op + d) = float2{o[0][r], o[1][r]};
      } else {
        *(f32x4 *)(op + d) = f32x4{o[0][r], o[1][r], o[2][r], o[3][r]};
      }
    }
    if (j == 0) *(float2 *)(part_ml + 2 * pbase) = float2{m, l};
  } else if (valid) {
    const float inv = 1.0f / l;
    float *op = out + qo_off;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int d = NT * (8 * (r >> 2) + 4 * j + (r & 3));
      if (PAD && d >= vhd) continue;  // (the width is a multiple of 4 and d of NT = 2 or 4: a store lies inside or outside as a whole)
      if constexpr (NT == 2) {
        *(float2 *)(op + d) = float2{o[0][r] * inv, o[1][r] * inv};
      } else {
        *(f32x4 *)(op + d) = f32x4{o[0][r] * inv, o[1][r] * inv, o[2][r] * inv, o[3][r] * inv};
      }
    }
  }
}

// (three workgroups of four wavefronts on a compute unit where the registers allow: 8192 rows, 32 / 8 heads of 64,
// 1377 -> 1324 us)
template <int HD, bool SPLIT, int G, bool PAD, bool BIAS = false>
__global__ __launch_bounds__(256 * G, G == 1 ? (HD == 64 && !PAD ? 3 : 2) : 1) void prefill_mfma_kernel(const float *__restrict__ q_rot,
                                                              const float *__restrict__ kc,
                                                              const float *__restrict__ vc,
                                                              float *__restrict__ out,
                                                              float *__restrict__ part_o,
                                                              float *__restrict__ part_ml, SeqTable st,
                                                              Shape sh, int ns, float c, DistanceBias db) {
  prefill_block<HD, SPLIT, G, PAD, BIAS>(blockIdx.x, q_rot, kc, vc, out, part_o, part_ml, st, sh, ns, c, db);
}

// For launches of two or three row blocks per compute unit: a workgroup takes, in turn, block b
// of the launch (blocks are numbered by decreasing key range), block 2N - 1 - b and block
// 2N + b (N workgroups): long, short and shorter ones that add up to about the same work for
// every workgroup, instead of the dispatcher starting another workgroup where one has ended
// (3.5 us later, measured).
template <int HD, int G, bool PAD, bool BIAS = false>
__global__ __launch_bounds__(256 * G, 1) void prefill_turns_kernel(const float *__restrict__ q_rot,
                                                                   const float *__restrict__ kc,
                                                                   const float *__restrict__ vc,
                                                                   float *__restrict__ out, SeqTable st, Shape sh,
                                                                   int n_blocks, float c, DistanceBias db) {
  const int N = gridDim.x, b = blockIdx.x;
  for (int turn = 0; turn < 3; ++turn) {
    const int bid = (turn & 1) ? (turn + 1) * N - 1 - b : turn * N + b;
    if (bid >= n_blocks) continue;
    if (turn) __syncthreads();  // the LDS stages are free: nobody is still merging the last block's halves
    prefill_block<HD, false, G, PAD, BIAS>(bid, q_rot, kc, vc, out, nullptr, nullptr, st, sh, 1, c, db);
  }
}

// Merge the key chunks of one (row block, kv head): online-softmax combine per row.
// Four workgroups per block (32 of its 128 virtual rows each, blockIdx.y) and up to eight
// chunks' loads in flight per thread: the kernel is bound by load latency, not by bytes.
__global__ __launch_bounds__(256) void prefill_combine_kernel(const float *__restrict__ part_o,
                                                              const float *__restrict__ part_ml,
                                                              float *__restrict__ out, SeqTable st, Shape sh,
                                                              int ns, float c, int tile_hd, int hd) {
  // hd: floats per row of the result; tile_hd: floats per row of a partial (the head dimension the tiles were laid out for)
  const int kvh = blockIdx.x % sh.KV, item = blockIdx.x / sh.KV;
  int s, vb;
  locate_block(st, item, s, vb);
  const int g = sh.g, hd4 = hd >> 2;
  const int VR = st.n_new[s] * g;
  const long long base = ((long long)item * sh.KV + kvh) * ns * 128;
  for (int idx = threadIdx.x; idx < 32 * hd4; idx += 256) {
    const int vl = blockIdx.y * 32 + idx / hd4, d4 = idx % hd4;
    const int v = vb * 128 + vl;
    if (v >= VR) continue;
    const int row = v / g, hg = v - row * g;
    float mm = -INFINITY;
    for (int k0 = 0; k0 < ns; k0 += 8) {
      float mk[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) mk[u] = part_ml[2 * (base + (long long)min(k0 + u, ns - 1) * 128 + vl)];
#pragma unroll
      for (int u = 0; u < 8; ++u) mm = fmaxf(mm, mk[u]);
    }
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    float ls = 0.f;
    for (int k0 = 0; k0 < ns; k0 += 8) {
      f32x4 x[8];
      float mk[8], lk[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const long long pi = base + (long long)min(k0 + u, ns - 1) * 128 + vl;
        x[u] = *(const f32x4 *)(part_o + pi * tile_hd + 4 * d4);
        mk[u] = part_ml[2 * pi];
        lk[u] = part_ml[2 * pi + 1];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        if (k0 + u >= ns) break;  // (repeats of the last chunk: 0 times what is not finite would not be 0)
        const float f = fast_exp2((mk[u] - mm) * c);  // 0 for a chunk that saw no visible key
        acc += f * x[u];
        ls += f * lk[u];
      }
    }
    *(f32x4 *)(out + ((long long)(st.tok_off[s] + row) * sh.H + kvh * g + hg) * hd + 4 * d4) = acc * (1.0f / ls);
  }
}

// ---------------------------------------------------------------------------
// Any head_dim: one wavefront per (row, head) and 256 columns of the values (blockIdx.z), lane = key for the
// scores, lane = d for the output.
__global__ __launch_bounds__(64) void generic_attn_kernel(const float *__restrict__ q_rot,
                                                          const float *__restrict__ kc,
                                                          const float *__restrict__ vc,
                                                          float *__restrict__ out, SeqTable st, Shape sh,
                                                          float scale, DistanceBias db) {
  extern __shared__ float smem[];
  const int hd = sh.hd, vhd = db.tab ? db.v_hd : hd;
  float *q_s = smem, *p_s = smem + hd;
  const int token = blockIdx.x, h = blockIdx.y, lane = threadIdx.x, v0 = blockIdx.z * 256;
  const int s = find_seq(st, token, st.tok_off);
  const int visible = st.start_pos[s] + (token - st.tok_off[s]) + 1;
  const int kvh = h / sh.g;
  const long long head_row = ((long long)st.slot[s] * sh.KV + kvh) * sh.cap;
  const float *kbase = kc + head_row * hd, *vbase = vc + head_row * vhd;
  const long long qo = ((long long)token * sh.H + h) * vhd;
  const float *q = q_rot + (db.tab ? token * db.q_stride + (long long)h * hd : qo);
  for (int d = lane; d < hd; d += 64) q_s[d] = q[d];
  __syncthreads();
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  for (int j0 = 0; j0 < visible; j0 += 64) {
    const int jj = j0 + lane;
    float sv = -INFINITY;
    if (jj < visible) {
      const float *kr = kbase + (long long)jj * hd;
      float dot = 0.f;
      for (int d = 0; d < hd; ++d) dot += q_s[d] * kr[d];
      sv = dot * scale;
      const int back = visible - 1 - jj;
      if (db.tab && back < db.reach) sv += db.tab[(long long)h * db.stride + (db.origin - back)] * 0.6931471805599453f;
    }
    float mx = sv;
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    const float mnew = fmaxf(m, mx);
    const float alpha = expf(m - mnew);
    const float p = expf(sv - mnew);
    float ps = p;
    for (int o = 32; o > 0; o >>= 1) ps += __shfl_xor(ps, o);
    l = l * alpha + ps;
    m = mnew;
    p_s[lane] = p;
    __syncthreads();
    const int cnt = min(64, visible - j0);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int d = v0 + lane + 64 * u;
      if (d < vhd) {
        float a = acc[u] * alpha;
        for (int t = 0; t < cnt; ++t) a += p_s[t] * vbase[(long long)(j0 + t) * vhd + d];
        acc[u] = a;
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int d = v0 + lane + 64 * u;
    if (d < vhd) out[qo + d] = acc[u] / l;
  }
}

constexpr float kLog2e = 1.4426950408889634f;

}  // namespace

bool decode_entries(const SeqTable &st, const Shape &sh, SeqTable &out) {
  if (sh.g < 1 || sh.g > 16) return false;
  const int per = 16 / sh.g;  // rows whose columns fill one tile
  memset(&out, 0, sizeof out);
  int n = 0;
  for (int s = 0; s < st.n_seqs; ++s) {
    const int groups = (st.n_new[s] + per - 1) / per;
    if (groups > 2 || n + groups > kMaxSeqs) return false;
    for (int k = 0; k < groups; ++k, ++n) {
      const int first = k * per, rows = st.n_new[s] - first < per ? st.n_new[s] - first : per;
      out.slot[n] = st.slot[s];
      out.start_pos[n] = st.start_pos[s] + first;  // the rows before them are in the cache already
      out.n_new[n] = rows;
      out.tok_off[n] = st.tok_off[s] + first;
    }
  }
  out.n_seqs = n;
  out.tok_off[n] = st.tok_off[st.n_seqs];
  return true;
}

int prefill_tile_head_dim(int hd) {
  if (hd < 4 || (hd & 3) || hd > 128) return 0;
  return hd <= 64 ? 64 : 128;
}

static int widest(const Shape &sh, int v_hd) { return v_hd > sh.hd ? v_hd : sh.hd; }

Path choose_path(const SeqTable &st, const Shape &sh, int v_hd) {
  // a few new rows per sequence: rows x heads of a group fit the 16 columns of the split-K
  // kernel's MFMA tiles, which then streams K and V once for all of them; up to twice as many
  // rows go to it as two entries (decode_entries), which still beats the key-chunked prefill.
  // Its tiles take any head dimension up to 256 that is a multiple of 4 (padded to 64, 128 or 256).
  SeqTable tmp;
  const bool v_ok = (v_hd & 3) == 0;  // (0 or the width of the value rows)
  if (v_ok && decode_tile_head_dim(sh.hd) && decode_tile_head_dim(widest(sh, v_hd)) && decode_entries(st, sh, tmp))
    return Path::kDecodeSplitK;
  // the MFMA prefill kernel's tiles: head dimensions up to 128 (padded to 64 or 128)
  if (!v_ok || !prefill_tile_head_dim(sh.hd) || !prefill_tile_head_dim(widest(sh, v_hd))) return Path::kGeneric;
  return Path::kPrefillMfma;
}

int plan_work(SeqTable &st, const Shape &sh, Path path) {
  st.work_off[0] = 0;
  for (int s = 0; s < st.n_seqs; ++s) {
    int items;
    if (path == Path::kPrefillMfma)
      items = (st.n_new[s] * sh.g + 127) / 128;
    else
      items = st.n_new[s];
    st.work_off[s + 1] = st.work_off[s] + items;
  }
  const int total = st.work_off[st.n_seqs];
  if (path == Path::kPrefillMfma) {
    // the prefill kernel wants per-sequence block counts and the sequences sorted by them
    for (int s = 0; s < st.n_seqs; ++s) st.work_off[s] = st.work_off[s + 1] - st.work_off[s];
    for (int s = 0; s < st.n_seqs; ++s) st.ord[s] = s;
    for (int a = 1; a < st.n_seqs; ++a)  // insertion sort, descending, stable
      for (int b = a; b > 0 && st.work_off[st.ord[b]] > st.work_off[st.ord[b - 1]]; --b) {
        const int t = st.ord[b];
        st.ord[b] = st.ord[b - 1];
        st.ord[b - 1] = t;
      }
  }
  return total;
}

static bool table_ok(const SeqTable &st, const Shape &sh) {
  if (st.n_seqs < 1 || st.n_seqs > kMaxSeqs || sh.g < 1 || sh.H != sh.KV * sh.g) return false;
  for (int s = 0; s < st.n_seqs; ++s)
    if (st.n_new[s] < 1 || st.start_pos[s] < 0 || st.start_pos[s] + st.n_new[s] > sh.cap || st.slot[s] < 0)
      return false;
  return true;
}

int prefill_key_splits(const SeqTable &st, const Shape &sh, int items) {
  const long long wgs = (long long)items * sh.KV;
  if (wgs >= 384) return 1;
  int longest = 0;  // key tiles of the longest row block
  for (int s = 0; s < st.n_seqs; ++s) {
    const int t = (st.start_pos[s] + st.n_new[s] + 31) / 32;
    longest = t > longest ? t : longest;
  }
  int ns = (int)((512 + wgs - 1) / wgs);
  // With long key ranges, about 1024 workgroups: four-wavefront workgroups that share the
  // compute units two or more at a time and drift apart then do better than 512 of eight
  // wavefronts, one per unit, whose two wavefronts per SIMD move in step (512 rows on 16384
  // cached, 128 row blocks: 1078 -> 1053 us); chunks under 32 tiles lose more to their set-up
  // (1024 rows into an empty cache: 109 -> 115 us).
  const int ns_1024 = (int)((1024 + wgs - 1) / wgs);
  if (longest / ns_1024 >= 32) ns = ns_1024;
  const int cap = longest / 8;  // at least eight key tiles per chunk
  if (ns > cap) ns = cap;
  if (ns > 16) ns = 16;
  return ns < 1 ? 1 : ns;
}

size_t prefill_partial_floats(const Shape &sh, int items, int ns, int v_hd) {
  return ns > 1 ? (size_t)items * sh.KV * ns * 128 * (prefill_tile_head_dim(widest(sh, v_hd)) + 2) : 0;
}

PrefillLaunch plan_prefill_launch(const Shape &sh, int items, int ns, int wgs_per_cu, int groups, int v_hd) {
  PrefillLaunch p;
  p.n_wgs = (long long)items * sh.KV * ns;
  // With fewer workgroups than three per compute unit everything is resident at
  // once: run one workgroup per compute unit (below) and give it eight wavefronts,
  // two per SIMD (G = 2).  Larger launches already have several workgroups per unit.
  p.groups = groups == 1 || groups == 2 ? groups : (p.n_wgs <= 768 ? 2 : 1);
  // static LDS of the kernel: `groups` K tiles and V tiles
  const int tile_hd = prefill_tile_head_dim(widest(sh, v_hd));
  const size_t static_lds = (size_t)16 * p.groups * (tile_hd == 64 ? TileUnits<64>::kTile : TileUnits<128>::kTile);
  p.pad = 0;
  // With fewer workgroups than three per compute unit everything is resident at
  // once and the dispatcher cannot balance the triangular work: one workgroup per
  // compute unit lets it hand the short row blocks to whichever unit finishes first.
  if (wgs_per_cu == 0 && p.n_wgs <= 768) wgs_per_cu = 1;
  p.wgs_per_cu = wgs_per_cu >= 1 && wgs_per_cu <= 3 ? wgs_per_cu : 0;
  if (p.wgs_per_cu) {
    const size_t want = (size_t)160 * 1024 / wgs_per_cu;  // one more workgroup would not fit
    const size_t floor_ = (size_t)160 * 1024 / (wgs_per_cu + 1) + 256;
    if (static_lds < floor_ && floor_ <= want) p.pad = floor_ - static_lds;
  }
  static const bool turns_off = getenv("SHAINET_HIP_PREFILL_NO_TURNS") != nullptr;
  // Turns only when the blocks fill them: otherwise compute units would stand idle where the
  // dispatcher's own hand-out keeps them busy (12 % slower at 640 blocks)
  const int turns = (int)((p.n_wgs + 255) / 256);
  p.turns = !turns_off && ns == 1 && p.groups == 2 && p.n_wgs > 256 && p.n_wgs <= 768 &&
                    p.n_wgs * 100 >= (long long)turns * 256 * 97
                ? turns
                : 0;
  return p;
}

hipError_t launch_prefill(const float *q_rot, const float *kc, const float *vc, float *out, float *partials,
                          const SeqTable &st, const Shape &sh, int items, int ns, float scale,
                          hipStream_t stream, int wgs_per_cu, int groups_wanted, hipEvent_t before, hipEvent_t after,
                          const DistanceBias *bias) {
  const DistanceBias db = bias ? *bias : DistanceBias{};
  const int v_hd = bias ? db.v_hd : sh.hd;
  const int tile_hd = prefill_tile_head_dim(widest(sh, v_hd));
  if (bias && (!db.tab || (v_hd & 3) || (db.q_stride & 3) || v_hd < 4 || (long long)sh.cap * v_hd * 4 > 0xffffffffLL)) return hipErrorInvalidValue;
  if (!table_ok(st, sh) || !tile_hd || !prefill_tile_head_dim(sh.hd) || items < 1 || ns < 1 || (ns > 1 && !partials)) return hipErrorInvalidValue;
  const bool pad = tile_hd != sh.hd;
  const PrefillLaunch plan = plan_prefill_launch(sh, items, ns, wgs_per_cu, groups_wanted, v_hd);
  const long long n_wgs = plan.n_wgs;
  if (n_wgs > 0x7fffffffLL) return hipErrorInvalidValue;
  // the kernels address a row of a (sequence, kv head) by a 32-bit byte offset from its first row
  if ((long long)sh.cap * sh.hd * 4 > 0xffffffffLL) return hipErrorInvalidValue;
  const float c = scale * kLog2e;
  dim3 grid((unsigned)n_wgs);
  float *part_o = partials;
  float *part_ml = partials ? partials + (size_t)items * sh.KV * ns * 128 * tile_hd : nullptr;
  const int groups = plan.groups;
  const size_t lds_pad = plan.pad;
  if (plan.turns) {
    const int turns = plan.turns;
    dim3 fewer((unsigned)((n_wgs + turns - 1) / turns));
#define SHAINET_LAUNCH_TURNS(HD_, ...)                                                                          \
  SHAINET_LAUNCH_TIMED((prefill_turns_kernel<HD_, 2, __VA_ARGS__>), fewer, dim3(512), 0, stream, before, after, q_rot, kc, \
                       vc, out, st, sh, (int)n_wgs, c, db)
    if (tile_hd == 64) {
      if (bias)
        SHAINET_LAUNCH_TURNS(64, true, true);
      else if (pad)
        SHAINET_LAUNCH_TURNS(64, true);
      else
        SHAINET_LAUNCH_TURNS(64, false);
    } else {
      if (bias)
        SHAINET_LAUNCH_TURNS(128, true, true);
      else if (pad)
        SHAINET_LAUNCH_TURNS(128, true);
      else
        SHAINET_LAUNCH_TURNS(128, false);
    }
#undef SHAINET_LAUNCH_TURNS
    return hipGetLastError();
  }
  hipEvent_t main_after = ns == 1 ? after : nullptr;  // with key chunks the combine kernel ends the timed stretch
#define SHAINET_LAUNCH_PREFILL(HD_, SPLIT_, ...)                                                               \
  do {                                                                                                          \
    if (groups == 2)                                                                                            \
      SHAINET_LAUNCH_TIMED((prefill_mfma_kernel<HD_, SPLIT_, 2, __VA_ARGS__>), grid, dim3(512), lds_pad, stream, before, \
                           main_after, q_rot, kc, vc, out, part_o, part_ml, st, sh, ns, c, db);                     \
    else                                                                                                        \
      SHAINET_LAUNCH_TIMED((prefill_mfma_kernel<HD_, SPLIT_, 1, __VA_ARGS__>), grid, dim3(256), lds_pad, stream, before, \
                           main_after, q_rot, kc, vc, out, part_o, part_ml, st, sh, ns, c, db);                     \
  } while (0)
#define SHAINET_LAUNCH_PREFILL_HD(HD_, ...)             \
  do {                                                  \
    if (ns > 1)                                         \
      SHAINET_LAUNCH_PREFILL(HD_, true, __VA_ARGS__);   \
    else                                                \
      SHAINET_LAUNCH_PREFILL(HD_, false, __VA_ARGS__);  \
  } while (0)
  if (tile_hd == 64) {
    if (bias)
      SHAINET_LAUNCH_PREFILL_HD(64, true, true);
    else if (pad)
      SHAINET_LAUNCH_PREFILL_HD(64, true);
    else
      SHAINET_LAUNCH_PREFILL_HD(64, false);
  } else {
    if (bias)
      SHAINET_LAUNCH_PREFILL_HD(128, true, true);
    else if (pad)
      SHAINET_LAUNCH_PREFILL_HD(128, true);
    else
      SHAINET_LAUNCH_PREFILL_HD(128, false);
  }
#undef SHAINET_LAUNCH_PREFILL_HD
#undef SHAINET_LAUNCH_PREFILL
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || ns == 1) return e;
  hipEvent_t none = nullptr;
  SHAINET_LAUNCH_TIMED(prefill_combine_kernel, dim3((unsigned)(items * sh.KV), 4), dim3(256), 0, stream, none, after,
                       part_o, part_ml, out, st, sh, ns, 1.0f, tile_hd, v_hd);  // the partials' maxima are already in log2 units
  return hipGetLastError();
}

hipError_t launch_generic(const float *q_rot, const float *kc, const float *vc, float *out,
                          const SeqTable &st, const Shape &sh, int total_tokens, float scale,
                          hipStream_t stream, const DistanceBias *bias) {
  const DistanceBias db = bias ? *bias : DistanceBias{};
  const int v_hd = bias ? db.v_hd : sh.hd;
  if (!table_ok(st, sh) || sh.hd < 1 || sh.hd > 8192 || v_hd < 1 || v_hd > 8192 || total_tokens < 1 || (bias && !db.tab))
    return hipErrorInvalidValue;
  const size_t smem = (size_t)(sh.hd + 64) * sizeof(float);
  hipLaunchKernelGGL(generic_attn_kernel, dim3((unsigned)total_tokens, (unsigned)sh.H, (unsigned)((v_hd + 255) / 256)), dim3(64),
                     smem, stream, q_rot, kc, vc, out, st, sh, scale, db);
  return hipGetLastError();
}

}  // namespace shainet
