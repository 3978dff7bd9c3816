// Causal grouped-query attention over the device KV cache for gfx950 (CDNA4).
//
// Together with decode_kernel.hip (one new row per sequence) these kernels replace
// attention_heads_cpu (llama_block.cr:302-401) and the reference's
// attention_kv_kernel (cuda_kernels.cu:734-806):
//
//   prefill_mfma_kernel   many new rows.  Query rows and the heads of a group
//       are flattened into "virtual rows"; a wavefront owns 32 of them.
//       K/V tiles of 32 keys are split into bf16 parts on their way
//       to LDS and consumed by v_mfma_f32_16x16x32_bf16.
//   generic_attn_kernel   any head_dim; one wavefront per (row, head).  Used for
//       head dims other than 64 and 128.
//
// The MFMA kernels compute S^T = K Q^T so that the probabilities come out of the MFMA
// accumulator already laid out as the B operand of O^T = V^T P^T: no transpose,
// no LDS round trip for P.  The contraction index of an MFMA may be visited in
// any order as long as A and B agree.
#include "attn_kernels.hpp"
#include "lane_quarters.hpp"
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
// Prefill: MFMA 16x16x32, K/V tiles staged through LDS.
//
// Virtual row v of a (sequence, kv head): query row v / g, head kvh*g + v % g.
// MFMA layout (lane l, j = l/16): A[m = l%16][k = 8j .. 8j+7], B[k = 8j .. 8j+7][n = l%16],
// D[m = 4j + r][n = l%16] for accumulator register r = 0..3.  A wavefront's 32 keys x 32 virtual rows are
// two blocks by two:
//   scores:  m = key within the block, n = virtual row, k = d.
//   output:  block t, m = d index (d = NT*m + t), contraction over the tile's 32 keys in
//            the order the score accumulators hold them.
// Row block number `rank` in dispatch order -> (sequence, block).  Level 0 is every
// sequence's last block (the longest key range), level 1 the one before, and so
// on.  st.work_off[s] = row blocks of sequence s, st.ord = sequences by descending
// block count.
// PER: blocks that are handed out together, those of one sequence from PER vb on.
template <int PER = 1>
__device__ __forceinline__ void locate_block(const SeqTable &st, int rank, int &s, int &vb) {
  auto count = [&](int i) { return (st.work_off[i] + PER - 1) / PER; };
  s = 0;
  int level = 0;
  for (int b = st.n_seqs - 1; b >= 0; --b) {  // levels [n_{b+1}, n_b) have b+1 active sequences
    const int lo = b + 1 < st.n_seqs ? count(st.ord[b + 1]) : 0;
    const int cnt = (count(st.ord[b]) - lo) * (b + 1);
    if (rank < cnt) {
      level = lo + rank / (b + 1);
      s = st.ord[rank % (b + 1)];
      break;
    }
    rank -= cnt;
  }
  vb = count(s) - 1 - level;
}

// The number of a block (PER = 1) in that order: all blocks of lower levels and those of its own level in front of it.
__device__ __forceinline__ int block_rank(const SeqTable &st, int s, int vb) {
  const int level = st.work_off[s] - 1 - vb;
  int rank = 0;
  bool before = true;
  for (int b = 0; b < st.n_seqs; ++b) {
    before = before && st.ord[b] != s;
    rank += min(st.work_off[st.ord[b]], level) + (before && st.work_off[st.ord[b]] > level ? 1 : 0);
  }
  return rank;
}

// Units of 16 bytes (eight bf16, one MFMA operand of a lane) that one key tile takes in LDS.  K: [part][octet of
// d][key], key r of octet o at place r ^ o % 8.  V: [part][group of eight keys][column], column d at place d / NT of block d % NT; group
// j holds the keys 4 j + {0 .. 3, 16 .. 19}, the ones whose probabilities the lanes of quarter j have.
// LDS serves a read in four turns of 16 lanes (0 .. 3, 12 .. 15, 20 .. 23 and 24 .. 27 are the first), whose units have to differ modulo 16: octets
// and groups are multiples of 16 apart, and only the lowest bits of a place depend on the octet of a quarter.  (33 units an octet, 72 or 136 a group: a third
// to half of all cycles of LDS were conflicts.)  So have 16 neighbouring threads' writes: eight octets of two keys eight apart, 16 columns.
template <int HD>
struct TileUnits {
  static constexpr int NT = HD / 16;
  static constexpr int kPartK = HD / 8 * 32;
  static constexpr int kBlockV = NT == 8 ? 18 : 20, kGroupV = NT * kBlockV, kPartV = 4 * kGroupV;
  static constexpr int kK = 3 * kPartK, kTile = kK + 3 * kPartV;
  static __device__ __forceinline__ int key_unit(int oct, int r) { return oct * 32 + (r ^ (oct & 7)); }
};

// Eight wavefronts, two groups of four, one of each on a SIMD and half a step apart: while one group has MFMAs, the
// other has softmax, splits and staging.
// G = 2: wavefronts 4..7 own the same 128 virtual rows as 0..3 and take every second key tile; the two
// halves merge through LDS.
// G = 1: two row blocks of a sequence; both groups walk the same key tiles, which are staged and split once for 256 rows.
// G = 3: one group, one row block; two or three such workgroups share a compute unit.
// One workgroup's work: the row block, or pair of them (and key chunk) number `bid` of the launch.
// PAD: the head dimension of the data (sh.hd, a multiple of 4) is smaller than HD, the one the
// tiles are laid out for: query elements beyond it are zeros (whatever stands in for the keys'
// there does not reach the scores), output elements beyond it are not stored, and a tile's
// pieces beyond it repeat the row's first piece (a cache hit, no HBM traffic).
// BIAS (with PAD): scores gain a value by distance (DistanceBias), value rows have a width of their own.
//
// Queries, keys, values and probabilities enter the MFMAs as exact sums of three bf16 numbers
// (split_mfma.hpp): the queries once, a key tile by the workgroup on its way to LDS, the probabilities in
// the registers the scores came in.  A tile costs a wavefront HD / 16 x 12 + HD / 16 x 12 MFMAs of 16 cycles (64:
// 1536) where the fp32 instruction took HD x 64 (4096).
// Us, v_mfma_f32_32x32x16_bf16 with both wavefronts of a SIMD in step | this: 2048 rows, 32 / 8 heads of 64, 108.5 | 97.6, 4096 rows 374 | 309, 512 rows on
// 16384 369 | 308; 512 rows on 16384, 32 / 4 heads of 128, 700 | 558, 2048 rows, 32 / 8 heads of 128, 222 | 194, 4096 rows 748 | 601; 2048 rows of 32 heads of 96
// 216 | 187; 32 / 8 heads of 64, 45 rows 12.4 | 11.7 (G = 3); 600 and 700 rows 33.1 | 34.2 and 36.1 | 36.6 one after the other (start and end of a workgroup, which leaves the
// compute units that it does not need to others: 17.3 | 12.2 and 21.7 | 21.7 among calls of other contexts).  Errors against 64 bits: below, at kTwoSums.
// What each part of it gave: half a step apart 104 | 100 and fragments a block ahead of their MFMAs 98; the layout of LDS without conflicts 96 | 92.6; a block's
// products on one accumulator rather than two in turn 1 %; two row blocks a workgroup and the queries' third parts in LDS 656 | 568 (512 rows on 16384, heads of 128).  In step
// again (no group waits half a step at the start) short ranges take 2 to 10 % longer.
// Registers: none spilled but for heads of 128 in turns (11, of padded tiles 14, with values by distance 33), with values by distance (2 to 20) and in padded tiles of G = 3
// (2); mostly where a row block begins and ends (in the blocks of code that hold the MFMAs: none in turns, 2 or 3 accesses a tile with values by distance, 1 in padded G = 3).
// What bounds it: heads of 128 the power the card may draw (matrix cores busy 78 % at 1.9 GHz); heads of 64 vector instructions: 281 and 16
// exponentials a tile and wavefront, of which a SIMD issues two during an MFMA of 16 cycles.  (Queries and keys as two fp16 numbers and scores of three products
// took 14 and 17 % less, but such numbers leave out up to 2^-21 of a product, and where a key's second parts have the signs of the
// query's that adds up.)
// Heads of 128 have no registers for the queries' third parts, or those of 24 of 32 octets: these lie in LDS, too.  (G = 2: both groups have the same.)
// G = 3: heads of 64 keep within 168 registers so (three wavefronts on a SIMD); heads of 128 those of 24, or two workgroups would not fit.
template <int HD, int G>
constexpr int kThirds = HD == 128 ? (G == 2 ? 4 : 3) : G == 3 ? 2 : 0;
// In LDS: the tiles' stages, behind them a wavefront's queries after another's.
template <int HD, int G>
constexpr int kThirdsAt = (G == 3 ? 1 : 2) * TileUnits<HD>::kTile;
template <int HD, int G>
constexpr int kLdsUnits = kThirdsAt<HD, G> + (G == 1 ? 8 : 4) * kThirds<HD, G> * 128;
static_assert(kLdsUnits<128, 1> * 16 <= 160 * 1024 && kLdsUnits<128, 2> * 16 <= 160 * 1024, "LDS of a compute unit");
static_assert(2 * kLdsUnits<128, 3> * 16 <= 160 * 1024, "two workgroups of one group share a compute unit");

template <int HD, bool SPLIT, int G, bool PAD, bool BIAS>
__device__ __forceinline__ void prefill_block(const int bid, const float *__restrict__ q_rot,
                                              const float *__restrict__ kc, const float *__restrict__ vc,
                                              float *__restrict__ out, float *__restrict__ part_o,
                                              float *__restrict__ part_ml, const SeqTable &st, const Shape &sh,
                                              int ns, float c, const DistanceBias &db) {
  static_assert(PAD || !BIAS, "sizes of their own come with padding");
  using U = TileUnits<HD>;
  constexpr int KS = HD / 32;   // MFMA steps along d of the scores
  constexpr int NT = HD / 16;   // d blocks of the output
  // items per thread to stage a tile of K (or V): G = 2, the tile of its group; G = 1, the one that all share, heads of 64: K is the first
  // group's, V the second's
  constexpr int NI = G == 1 ? 1 : HD / 64;
  constexpr bool kOneOfTwo = G == 1 && HD == 64;
  __shared__ __attribute__((aligned(16))) u32x4 lds[kLdsUnits<HD, G>];

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
  locate_block<G == 1 ? 2 : 1>(st, item, s, vb);
  // These are the same for all lanes of a wavefront, which the compiler cannot see: said so,
  // tile counts, loop conditions and address bases live in scalar registers
  auto uniform = [](int x) { return __builtin_amdgcn_readfirstlane(x); };
  s = uniform(s);
  vb = uniform(vb);
  const int g = sh.g, T = st.n_new[s], S = st.start_pos[s];
  const int L = S + T, VR = T * g;
  const int lane = threadIdx.x & 63;
  const int wave = uniform((threadIdx.x >> 6) & 3);  // which 32 virtual rows of the block
  const int gidx = G == 3 ? 0 : uniform(threadIdx.x >> 8);  // which group of wavefronts
  const int wg_hi = st.start_pos[s] + min((vb + 1) * (G == 1 ? 256 : 128) - 1, st.n_new[s] * sh.g - 1) / sh.g;
  if (G == 1) vb = 2 * vb + gidx;
  constexpr int kStep = G == 2 ? 2 : 1;      // key tiles of a step
  const int first_tile = G == 2 ? gidx : 0;  // a group's first key tile
  const int n = lane & 15, j = lane >> 4;
  const int v0 = vb * 128 + wave * 32;
  const bool wave_active = v0 < VR;
  const int wave_lo = S + (wave_active ? v0 / g : 0);                 // smallest lim in the wavefront
  const int wave_hi = wave_active ? S + min(v0 + 31, VR - 1) / g : -1;  // largest
  const int n_tiles = wg_hi / 32 + 1;
  const int tiles_per_chunk = SPLIT ? (n_tiles + ns - 1) / ns : n_tiles;
  int kt0 = chunk * tiles_per_chunk;
  if constexpr (G == 3) asm volatile("" : "+s"(kt0));  // (of a range that begins at 0 it keeps addresses per thread: 28 spills in padded tiles, 159 | 114 us at 64 sequences of 100 rows)
  const int kt1 = min(n_tiles, kt0 + tiles_per_chunk);
  const int hd = PAD ? uniform(sh.hd) : HD;  // floats between two rows of q, K, V and the output
  const long long head_base = (long long)st.slot[s] * sh.seq_stride + (long long)kvh * sh.cap * hd;
  const float *kbase = kc + head_base;
  const int vhd = BIAS ? uniform(db.v_hd) : hd;
  const float *vbase = vc + (BIAS ? ((long long)st.slot[s] * sh.KV + kvh) * sh.cap * vhd : head_base);
  // a lane's two virtual rows, v0 + n and 16 on
  int lim[2];  // last visible key of the row
  long long q_off[2];        // of the row's query
  const float *bias_row[2];  // entry of key row k: bias_row[k]
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int my_v = v0 + 16 * b + n;
    const int row = my_v < VR ? my_v / g : T - 1, hg = my_v < VR ? my_v - row * g : 0;
    lim[b] = S + row;
    q_off[b] = BIAS ? (st.tok_off[s] + row) * db.q_stride + (long long)(kvh * g + hg) * hd
                    : ((long long)(st.tok_off[s] + row) * sh.H + kvh * g + hg) * hd;
    bias_row[b] = BIAS ? db.tab + (long long)(kvh * g + hg) * db.stride + (db.origin - lim[b]) : nullptr;
  }

  // what a thread stages of its group's tile: K, an octet of d of a row; V, eight rows of a column
  unsigned k_off[NI], v_off[NI];
  int k_row[NI], v_row[NI], k_unit[NI], v_unit[NI];
  bool k_second[NI];  // the octet's second half lies within the row
#pragma unroll
  for (int u = 0; u < NI; ++u) {
    const int idx = (G != 1 || kOneOfTwo ? threadIdx.x & 255 : threadIdx.x) + 256 * u;
    const int pair = HD == 128 ? idx >> 5 : idx >> 4;  // (of keys eight apart)
    const int oct = (idx & 7) | (HD == 128 ? idx >> 1 & 8 : 0), r = (idx & 8) | (pair & 7) | (pair & 8) << 1;
    k_row[u] = r;
    k_off[u] = PAD && 8 * oct >= hd ? 0u : 32u * oct;
    k_second[u] = !PAD || 8 * oct + 4 < hd;
    k_unit[u] = (G == 2 ? gidx * U::kTile : 0) + U::key_unit(oct, r);
    const int d = idx % HD, group = idx / HD;
    v_row[u] = 4 * group;
    v_off[u] = PAD && d >= vhd ? 0u : 4u * d;
    v_unit[u] = (G == 2 ? gidx * U::kTile : 0) + U::kK + group * U::kGroupV + d % NT * U::kBlockV + d / NT;
  }
  const unsigned k_stride = (unsigned)hd * 4, v_stride = (unsigned)vhd * 4;
  f32x4 stage_k[NI][2];
  float stage_v[NI][8];
  // a scalar base and a 32-bit byte offset per lane (a head's rows span less than 4 GiB: checked
  // at launch); rows past the last one repeat it
  auto load_k = [&](int sp) {
    if (kOneOfTwo && gidx) return;
    const int first = (kt0 + kStep * sp + first_tile) * 32;
#pragma unroll
    for (int u = 0; u < NI; ++u) {
      const char *p = (const char *)kbase + ((unsigned)min(first + k_row[u], L - 1) * k_stride + k_off[u]);
      stage_k[u][0] = *(const f32x4 *)p;
      stage_k[u][1] = *(const f32x4 *)(p + (k_second[u] ? 16 : 0));
    }
  };
  auto load_v = [&](int sp) {
    if (kOneOfTwo && !gidx) return;
    const int first = (kt0 + kStep * sp + first_tile) * 32;
    if (first + 32 <= L) {
      const char *base = (const char *)vbase + (unsigned long long)first * v_stride;
#pragma unroll
      for (int u = 0; u < NI; ++u) {
        const unsigned off = (unsigned)v_row[u] * v_stride + v_off[u];
#pragma unroll
        for (int i = 0; i < 8; ++i) stage_v[u][i] = *(const float *)(base + (unsigned long long)((i & 3) + 16 * (i >> 2)) * v_stride + off);
      }
    } else {
#pragma unroll
      for (int u = 0; u < NI; ++u)
#pragma unroll
        for (int i = 0; i < 8; ++i)
          stage_v[u][i] = *(const float *)((const char *)vbase +
                                           ((unsigned)min(first + v_row[u] + (i & 3) + 16 * (i >> 2), L - 1) * v_stride + v_off[u]));
    }
  };
  auto park_k = [&](int sp) {
    if (kOneOfTwo && gidx) return;
    u32x4 *const to = lds + (G == 1 && sp & 1 ? U::kTile : 0);
#pragma unroll
    for (int u = 0; u < NI; ++u) {
      u32x4 h, m, l;
      split_octet(stage_k[u][0], stage_k[u][1], h, m, l);
      to[k_unit[u]] = h;
      to[k_unit[u] + U::kPartK] = m;
      to[k_unit[u] + 2 * U::kPartK] = l;
    }
  };
  auto park_v = [&](int sp) {
    if (kOneOfTwo && !gidx) return;
    u32x4 *const to = lds + (G == 1 && sp & 1 ? U::kTile : 0);
#pragma unroll
    for (int u = 0; u < NI; ++u) {
      u32x4 h, m, l;
      split_octet(f32x4{stage_v[u][0], stage_v[u][1], stage_v[u][2], stage_v[u][3]},
                  f32x4{stage_v[u][4], stage_v[u][5], stage_v[u][6], stage_v[u][7]}, h, m, l);
      to[v_unit[u]] = h;
      to[v_unit[u] + U::kPartV] = m;
      to[v_unit[u] + 2 * U::kPartV] = l;
    }
  };

  // steps of a tile, or (G = 2) of one per group; below "tile sp" is a group's tile of step sp (in the last step the second group
  // may have none left: it stages its last rows again)
  const int n_sp = kt0 < kt1 ? (kt1 - kt0 + kStep - 1) / kStep : 0;
  if (n_sp > 0) {
    load_k(0);
    load_v(0);
  }
  // the row's query, scaled by scale * log2(e): scores come out in log2 units
  u32x4 qf[KS][2][3];
  u32x4 *const third = lds + kThirdsAt<HD, G> + (G == 1 ? 4 * gidx + wave : wave) * (kThirds<HD, G> * 128) + lane;
  bool apart;  // some query of the wavefront needs its scores in fp32
  {
    float least = INFINITY, most = 0.f;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      f32x4 t[KS][2];
      const float *qp = q_rot + q_off[b] + 8 * j;
#pragma unroll
      for (int i = 0; i < KS; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          // (lanes past the last virtual row repeat the last row: their results are never used)
          t[i][h] = f32x4{0.f, 0.f, 0.f, 0.f};
          if (!PAD || 32 * i + 8 * j + 4 * h < hd) t[i][h] = *(const f32x4 *)(qp + 32 * i + 4 * h);
        }
#pragma unroll
      for (int i = 0; i < KS; ++i) {
        split_octet(t[i][0] * c, t[i][1] * c, qf[i][b][0], qf[i][b][1], qf[i][b][2]);
        if (i < kThirds<HD, G> && (G != 2 || gidx == 0)) third[(2 * i + b) * 64] = qf[i][b][2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          if (PAD && 32 * i + 8 * j + 4 * h >= hd) continue;
#pragma unroll
          for (int w = 0; w < 4; ++w) {
            const float size = fabsf(t[i][h][w] * c);
            least = fminf(least, size);
            most = fmaxf(most, size);
          }
        }
      }
    }
    apart = false;
    // (looked at closely only where there is a zero or something out of the ordinary)
    if (__builtin_expect(__any(!(least >= 0x1p-109f) || !(most < 0x1p100f)), 0)) {
      QueryRange range;
#pragma clang loop unroll(disable)
      for (int d = 4 * j; d < hd; d += 16) {
        range.add(*(const f32x4 *)(q_rot + q_off[0] + d));
        range.add(*(const f32x4 *)(q_rot + q_off[1] + d));
      }
      apart = __any(range.apart(c));
    }
  }

  // Online softmax against a reference value per virtual row instead of the running maximum: m_ref is only moved
  // (and l, O rescaled) when a score exceeds it by more than kTau, or for a row's first visible key;
  // probabilities are then at most 2^kTau, no overflow.  A tile on the common path costs a maximum, 16
  // subtractions, exp2 and adds per lane.  (Sums of scores that begin at -m_ref save the subtractions, 1 to 2.6 %, but round more often where a
  // score is small beside m_ref: errors against 64 bits grew by 3 to 16 %.)
  constexpr float kTau = 8.f;
  float m_ref[2] = {0.f, 0.f}, l[2] = {0.f, 0.f};
  float thr[2] = {-INFINITY, -INFINITY};  // a row's scores move m_ref when above this: anything finite until its first key, m_ref + kTau after
  f32x4 o[NT][2];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int b = 0; b < 2; ++b) o[t][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  // O is a chain of sums, in which each of a tile's six products would be rounded to O's last place: twice the error of one rounding a tile (relative
  // to 64 bits, 400 rows on 4000, 32 / 8 heads of 64, 5.4e-7 | 2.8e-7; 512 on 4096, 32 / 4 heads of 128, 6.1e-7 | 3.6e-7).
  // kTwoSums: the five smaller products have a sum of their own, for which heads of 64 have the registers (2048 rows 97.4 | 97.6 us, 8192 rows 1156 | 1151).
  // kOwnSum: a tile's products are added up before they join O (a sum more beside each six MFMAs: heads of 128, 2048 rows 192 | 193.5 us, 800 rows 71.9 | 73.1).
  // Heads of 128 in two blocks a workgroup have neither: it would take 4 to 5 % (512 on 16384 558 | 586 us).  Nor have ranges of a few tiles.
  constexpr bool kTwoSums = HD == 64 && G != 3, kOwnSum = G == 3 ? SPLIT : HD == 128 && G == 2;
  f32x4 low[kTwoSums ? NT : 1][2];
#pragma unroll
  for (int t = 0; t < (kTwoSums ? NT : 1); ++t) low[t][0] = low[t][1] = f32x4{0.f, 0.f, 0.f, 0.f};
  // A step of a group has two halves: MFMAs (O^T += V^T(sp - 1) P^T(sp - 1), scores of tile sp) and everything else (softmax of tile sp, P
  // split, V(sp) and K(sp + 1) parked, the next requested), a barrier behind each.  The second group is half a step behind: while a SIMD's
  // one wavefront has MFMAs only, its other one has none.  G = 2: each group stages its own tiles, one of K and one of V.  G = 1: both stage
  // half of each, into two stages in turn; the second group does so a step ahead, for the first needs them half a step later.
  // (heads of 128, G = 2, have no registers for a tile of K during the MFMAs: it is requested and parked within the other half)
  constexpr bool kLate = HD == 128 && G != 1;
  const int k_at[2] = {U::key_unit(j, n) + (G == 2 ? gidx * U::kTile : 0), (U::key_unit(j, n) ^ 4) + (G == 2 ? gidx * U::kTile : 0)}, v_at = U::kK + j * U::kGroupV + n + (G == 2 ? gidx * U::kTile : 0);
  // tiles that some row of the wavefront sees
  const int n_mine = max(0, (min(kt1, wave_hi / 32 + 1) - kt0 - first_tile + kStep - 1) / kStep) * (wave_hi >= 0);
  constexpr bool kExact = G == 3;                 // nothing is requested for nobody: ranges are short
  constexpr bool kScoresFirst = HD == 128 || G == 3;  // in the loop below
  auto stage_v_tile = [&](int sp) {
    park_v(sp);
    if constexpr (!kLate) {
      if (!kExact || sp + 1 < n_sp) load_v(sp + 1);
    } else if (sp + 1 < n_sp) {
      load_k(sp + 1);
    }
  };
  auto stage_k_tile = [&](int sp) {
    if ((HD == 64 && !kExact) || sp + 1 < n_sp) {
      park_k(sp + 1);
      if constexpr (kLate) load_v(sp + 1);
    }
    if (!kLate && (!kExact || sp + 2 < n_sp)) load_k(sp + 2);
  };
  f32x4 p[2][2];   // [virtual rows][keys]: scores, then probabilities
  u32x4 pf[2][3];  // their parts
  f32x4 near_bias[BIAS ? 2 : 1][2];
  bool near = false;
  auto scores = [&](int sp) {
    const int kt = kt0 + kStep * sp + first_tile;
    auto key = [&](int k, int w) { return lds[k_at[k / 2 & 1] + (G == 1 && sp & 1 ? U::kTile : 0) + w * U::kPartK + k / 2 * 128 + k % 2 * 16]; };
    // the tile's values by distance are asked for in front of its MFMAs; a tile that lies
    // `reach` or more behind all rows of the wavefront has none
    if constexpr (BIAS) {
      near = wave_lo - (kt * 32 + 31) < db.reach;
      if (near) {
        struct __attribute__((packed, aligned(4))) Four { f32x4 v; };
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int a = 0; a < 2; ++a) near_bias[b][a] = ((const Four *)(bias_row[b] + kt * 32 + 16 * a + 4 * j))->v;
      }
    }
    // S^T of the key tile: 32 keys x 32 virtual rows; fragments arrive a block ahead of the MFMAs that take them
    u32x4 fr[2][3], qt[2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) p[b][a] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 3; ++w) fr[0][w] = key(0, w);
#pragma unroll
    for (int k = 0; k < 2 * KS; ++k) {
      const int i = k / 2, a = k % 2;
      if (i < kThirds<HD, G> && a == 0) {
#pragma unroll
        for (int b = 0; b < 2; ++b) qt[b] = third[(2 * i + b) * 64];
      }
      if (k + 1 < 2 * KS) {
#pragma unroll
        for (int w = 0; w < 3; ++w) fr[k + 1 & 1][w] = key(k + 1, w);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int w = 0; w < 6; ++w)
          p[b][a] = mfma_bf16_16(fr[k & 1][kPartA[w]], kPartB[w] == 2 && i < kThirds<HD, G> ? qt[b] : qf[i][b][kPartB[w]], p[b][a]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto softmax = [&](int sp) {
    const int kt = kt0 + kStep * sp + first_tile;
    if constexpr (BIAS) {
      if (near) {
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int a = 0; a < 2; ++a) p[b][a] += near_bias[b][a];
      }
    }
    if (kt * 32 + 31 > wave_lo) {  // tile crosses the diagonal for some row of this wavefront
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (kt * 32 + 16 * a + 4 * j + r > lim[b]) p[b][a][r] = -INFINITY;
    }
    float mx[2];
#pragma unroll
    for (int b = 0; b < 2; ++b)
      mx[b] = fmaxf(fmaxf(fmaxf(fmaxf(p[b][0][0], p[b][0][1]), p[b][0][2]), fmaxf(fmaxf(p[b][0][3], p[b][1][0]), p[b][1][1])),
                    fmaxf(p[b][1][2], p[b][1][3]));
    // mx covers this lane's quarter of the row's keys in the tile; the row's maximum is above thr
    // exactly when one of the four quarters' is (never for a row without a visible key here:
    // -inf), so the quarters only exchange their maxima once a move is certain
    if (__builtin_amdgcn_ballot_w64(mx[0] > thr[0] || mx[1] > thr[1]) != 0) {
      // rare after a row's first tiles: move the reference to this tile's maximum
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        mx[b] = max_across_quarters(mx[b]);
        if (mx[b] > thr[b]) {
          const float alpha = thr[b] != -INFINITY ? fast_exp2(m_ref[b] - mx[b]) : 1.f;  // nothing to rescale before a row's first key
          m_ref[b] = mx[b];
          thr[b] = mx[b] + kTau;
          l[b] *= alpha;
#pragma unroll
          for (int t = 0; t < NT; ++t) o[t][b] *= alpha;
          if constexpr (kTwoSums) {
#pragma unroll
            for (int t = 0; t < NT; ++t) low[t][b] *= alpha;
          }
        }
      }
    }
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      float psum = 0.f;
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          p[b][a][r] = fast_exp2(p[b][a][r] - m_ref[b]);
          psum += p[b][a][r];
        }
      l[b] += psum;
      split_octet(p[b][0], p[b][1], pf[b][0], pf[b][1], pf[b][2]);
    }
  };
  auto outputs = [&](int sp) {  // O^T += V^T P^T
    const u32x4 *const vl = lds + v_at + (G == 1 && sp & 1 ? U::kTile : 0);
    u32x4 fr[2][3];
    f32x4 before;  // (kOwnSum) the last block's sum, which joins O while the next one's MFMAs run
#pragma unroll
    for (int w = 0; w < 3; ++w) fr[0][w] = vl[w * U::kPartV];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      if (t + 1 < NT) {
#pragma unroll
        for (int w = 0; w < 3; ++w) fr[t + 1 & 1][w] = vl[w * U::kPartV + (t + 1) * U::kBlockV];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        if constexpr (kOwnSum) {
          f32x4 own = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int w = 0; w < 6; ++w) own = mfma_bf16_16(fr[t & 1][kPartA[w]], pf[b][kPartB[w]], own);
          if (t + b > 0) o[b ? t : t - 1][b ^ 1] += before;
          before = own;
        } else {
#pragma unroll
          for (int w = 0; w < 6; ++w) {
            f32x4 &to = kTwoSums && w < 5 ? low[t][b] : o[t][b];
            to = mfma_bf16_16(fr[t & 1][kPartA[w]], pf[b][kPartB[w]], to);
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (kOwnSum) o[NT - 1][1] += before;
  };
  if (n_sp > 0) {
    park_k(0);
    if (!kLate && (!kExact || n_sp > 1)) load_k(1);
  }
  __syncthreads();
  const bool half_apart = G == 1 || (G == 2 && n_sp > 1);  // (a tile each: 64 rows, 32 / 8 heads of 64, 14.0 | 13.4 us with both groups in step)
  if (gidx == 1 && half_apart) {
    if (G == 1 && n_sp > 0) {
      stage_v_tile(0);
      stage_k_tile(0);
    }
    __syncthreads();
  }
  const int ahead = G == 1 ? gidx : 0;
  // (what is requested and parked behind the last tile is nobody's: its rows are the last one again, its stage is free)
  int sp = 0;
  if constexpr (!kScoresFirst) {
    if (n_mine > 0) scores(0);
    for (; sp < n_mine - 1; ++sp) {
      __syncthreads();  // nobody of the group reads V(sp - 1) and K(sp) any more
      stage_v_tile(sp + ahead);
      softmax(sp);
      stage_k_tile(sp + ahead);
      __syncthreads();  // V(sp) and K(sp + 1) are there
      outputs(sp);
      scores(sp + 1);
    }
  } else {  // (a loop that begins with the scores has no spills here; heads of 64 take 2 % longer so)
    for (; sp < n_mine; ++sp) {
      __builtin_amdgcn_s_setprio(1);
      scores(sp);
      __builtin_amdgcn_s_setprio(0);
      __syncthreads();
      __builtin_amdgcn_sched_barrier(0);  // (V is split in this half; heads of 64 have fewer MFMAs than this half has work)
      stage_v_tile(sp + ahead);
      softmax(sp);
      if constexpr (kLate) __builtin_amdgcn_sched_barrier(0);  // (K is on its way meanwhile)
      stage_k_tile(sp + ahead);
      __syncthreads();
      __builtin_amdgcn_s_setprio(1);
      outputs(sp);
    }
    __builtin_amdgcn_s_setprio(0);
  }
  for (; sp < n_sp; ++sp) {  // the wavefront's last tile (heads of 64), and those that only others see
    __syncthreads();
    if (sp + ahead < n_sp) stage_v_tile(sp + ahead);
    if (!kScoresFirst && sp < n_mine) softmax(sp);
    if (sp + ahead + 1 < n_sp) stage_k_tile(sp + ahead);
    __syncthreads();
    if (!kScoresFirst && sp < n_mine) outputs(sp);
  }
  if (gidx == 0 && half_apart) __syncthreads();
  if constexpr (kTwoSums) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int b = 0; b < 2; ++b) o[t][b] += low[t][b];
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
    float probe = l[0] * 0.f + l[1] * 0.f, least = INFINITY;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        probe = fmaf(o[t][r >> 2][r & 3], 0.f, probe);
        least = fminf(least, fabsf(o[t][r >> 2][r & 3]));
      }
    bool again = apart || __any(probe != 0.f);
    float up = 1.f, down = 1.f;
    if (__builtin_expect(__any(least < 0x1p-80f && (thr[0] != -INFINITY || thr[1] != -INFINITY)), 0) && !again) {
      int tid = threadIdx.x;
      asm volatile("" : "+v"(tid));
      unsigned small = ~0u;  // (zeros lie above all)
#pragma clang loop unroll(disable)
      for (int kt = kt0 + first_tile; kt < kt1 && kt * 32 <= wave_hi; kt += kStep) {
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
      const int n = tid & 15, j = (tid & 63) >> 4;
      int lim[2];
      const float *bias_row[2], *qr[2];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int my_v = min(v0 + 16 * b + n, VR - 1), row = my_v / g, hg = my_v - row * g;
        lim[b] = S + row;
        qr[b] = q_rot + 4 * j + (BIAS ? (st.tok_off[s] + row) * db.q_stride + (long long)(kvh * g + hg) * hd
                                      : ((long long)(st.tok_off[s] + row) * sh.H + kvh * g + hg) * hd);
        bias_row[b] = BIAS ? db.tab + (long long)(kvh * g + hg) * db.stride + (db.origin - lim[b]) : nullptr;
        m_ref[b] = 0.f, l[b] = 0.f, thr[b] = -INFINITY;
      }
      f32x4 sum[NT][2];
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int b = 0; b < 2; ++b) sum[t][b] = f32x4{0.f, 0.f, 0.f, 0.f};
      // Tile by tile: scores from the fp32 instruction, lane quarter j with d = 16 i + 4 j .. + 3 of step i, here against
      // the running maximum; the products with V likewise where every row sees the whole tile, else key by key
      // (what a row does not see it does not multiply by zero either).
#pragma clang loop unroll(disable)
      for (int kt = kt0 + first_tile; kt < kt1 && kt * 32 <= wave_hi; kt += kStep) {
        const int first = kt * 32;
        const bool whole = first + 31 <= wave_lo;
        const float *kr[2] = {kbase + (long long)min(first + n, L - 1) * hd + 4 * j, kbase + (long long)min(first + 16 + n, L - 1) * hd + 4 * j};
        float p[2][8];  // [virtual rows][16 (i / 4) + 4 j + i % 4 of the keys]
        {
          f32x4 sc[2][2];
#pragma unroll
          for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int a = 0; a < 2; ++a) sc[b][a] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma clang loop unroll(disable)
          for (int d = 0; d < hd; d += 16) {
            const bool in = !PAD || d + 4 * j < hd;
            f32x4 kv[2], qv[2];
#pragma unroll
            for (int a = 0; a < 2; ++a) {
              kv[a] = in ? *(const f32x4 *)(kr[a] + d) : f32x4{0.f, 0.f, 0.f, 0.f};
              qv[a] = in ? *(const f32x4 *)(qr[a] + d) * c : f32x4{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
              for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int i = 0; i < 4; ++i) sc[b][a] = mfma_f32_16(kv[a][i], qv[b][i], sc[b][a]);
          }
#pragma unroll
          for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int i = 0; i < 8; ++i) p[b][i] = sc[b][i >> 2][i & 3];
        }
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          if (BIAS && wave_lo - (first + 31) < db.reach) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
              const int key = first + 16 * (i >> 2) + 4 * j + (i & 3);
              if (key <= lim[b] && lim[b] - key < db.reach) p[b][i] += bias_row[b][key];
            }
          }
          float mx = -INFINITY;
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            if (!whole && first + 16 * (i >> 2) + 4 * j + (i & 3) > lim[b]) p[b][i] = -INFINITY;
            mx = fmaxf(mx, p[b][i]);
          }
          mx = fmaxf(mx, __shfl_xor(mx, 16));
          mx = fmaxf(mx, __shfl_xor(mx, 32));
          if (mx > thr[b]) {
            const float alpha = thr[b] == -INFINITY ? 0.f : fast_exp2(thr[b] - mx);
            m_ref[b] = thr[b] = mx;
            l[b] *= alpha;
#pragma unroll
            for (int t = 0; t < NT; ++t) sum[t][b] *= alpha;
          }
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            p[b][i] = fast_exp2(p[b][i] - m_ref[b]);
            l[b] += p[b][i];
          }
        }
        if (whole) {
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const float *vr = vbase + (long long)(first + 16 * (i >> 2) + 4 * j + (i & 3)) * vhd;
#pragma unroll
            for (int w = 0; w < NT / 4; ++w) {
              const int d = NT * n + 4 * w;
              const f32x4 v = *(const f32x4 *)(vr + (PAD && d >= vhd ? 0 : d)) * up;
#pragma unroll
              for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int b = 0; b < 2; ++b) sum[4 * w + t][b] = mfma_f32_16(v[t], p[b][i], sum[4 * w + t][b]);
            }
          }
          continue;
        }
#pragma clang loop unroll(disable)
        for (int i = 0; i < 8; ++i) {
          const float own[2] = {p[0][0], p[1][0]};
#pragma unroll
          for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int k = 0; k < 7; ++k) p[b][k] = p[b][k + 1];  // (no register is indexed by a loop counter)
#pragma clang loop unroll(disable)
          for (int h = 0; h < 4; ++h) {
            const int key = first + 16 * (i >> 2) + 4 * h + (i & 3);
            const float e[2] = {__shfl(own[0], n + 16 * h), __shfl(own[1], n + 16 * h)};
            if (key > max(lim[0], lim[1])) continue;
            const float *vr = vbase + (long long)key * vhd;
#pragma unroll
            for (int w = 0; w < NT; ++w) {  // floats 4 w .. 4 w + 3 of the 4 NT columns that a lane holds
              const int d = NT * 4 * j + 4 * w;
              const f32x4 v = *(const f32x4 *)(vr + (PAD && d >= vhd ? 0 : d)) * up;
#pragma unroll
              for (int b = 0; b < 2; ++b) {
                if (key > lim[b]) continue;
#pragma unroll
                for (int k = 0; k < 4; ++k) sum[(4 * w + k) % NT][b][(4 * w + k) / NT] = fmaf(e[b], v[k], sum[(4 * w + k) % NT][b][(4 * w + k) / NT]);
              }
            }
          }
        }
      }
      // (one by one through registers of their own: as whole accumulators the loop above would move them about)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          float x = sum[t][r >> 2][r & 3] * down;
          asm volatile("" : "+v"(x));
          o[t][r >> 2][r & 3] = x;
        }
    }
  }

  // (what a lane works on is found again from its number: kept for here it would cost the loop above registers)
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  // what the merges below call the maximum: the reference the sums are relative to, in log2
  // units, or -inf for a row that saw no key (its l and O are 0)
  float m[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    l[b] = sum_across_quarters(l[b]);
    m[b] = thr[b] == -INFINITY ? -INFINITY : m_ref[b];
  }
  if constexpr (G == 2) {
    const int lane = tid & 63;
    // the second group hands its (max, sum, O) to the first through the tile stages
    f32x4 *xo = (f32x4 *)lds;                       // [4 row chunks][2 NT registers of four][64 lanes]
    float *xm = (float *)lds + 4 * 8 * NT * 64;     // [4][2][64] max, then the same of sums
    static_assert(sizeof lds >= (4 * 8 * NT * 64 + 1024) * sizeof(float), "the merge fits the tiles");
    __syncthreads();  // nobody reads tiles any more
    if (gidx == 1) {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
#pragma unroll
        for (int t = 0; t < NT; ++t) xo[((wave * NT + t) * 2 + b) * 64 + lane] = o[t][b];
        xm[(wave * 2 + b) * 64 + lane] = m[b];
        xm[512 + (wave * 2 + b) * 64 + lane] = l[b];
      }
    }
    __syncthreads();
    if (gidx == 1) return;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const float m1 = xm[(wave * 2 + b) * 64 + lane], l1 = xm[512 + (wave * 2 + b) * 64 + lane];
      const float mnew = fmaxf(m[b], m1);
      // a side that saw no visible key has max -inf: its factor is 0 (and both may be, in a key chunk)
      const float a0 = m[b] == -INFINITY ? 0.f : fast_exp2(m[b] - mnew);
      const float a1 = m1 == -INFINITY ? 0.f : fast_exp2(m1 - mnew);
#pragma unroll
      for (int t = 0; t < NT; ++t) o[t][b] = o[t][b] * a0 + xo[((wave * NT + t) * 2 + b) * 64 + lane] * a1;
      l[b] = l[b] * a0 + l1 * a1;
      m[b] = mnew;
    }
  }
  // A lane has 4 NT neighbouring columns of a row: stored as they are, an instruction would write 16 bytes into each of 64 lines.  Traded among the
  // quarters, four lanes write 64 bytes together (us, as they are | traded: 64 sequences of 64 rows, 32 / 8 heads of 64, 33.2 | 27.0, of 100 rows, 32 heads of
  // 128, 121 | 113, 64 sequences of 96 rows, two blocks a workgroup 58.2 | 52.7).
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int n = tid & 15, j = (tid & 63) >> 4, my_v = v0 + 16 * b + n;
    f32x4 line[NT / 4][4];  // [..][i]: the piece of four columns at NT i + 4 h + j
#pragma unroll
    for (int h = 0; h < NT / 4; ++h) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r = (4 * h + q) / (NT / 4), w = 4 * ((4 * h + q) % (NT / 4));
        line[h][q] = f32x4{o[w][b][r], o[w + 1][b][r], o[w + 2][b][r], o[w + 3][b][r]};
      }
      transpose_quarters(line[h]);
    }
    if (my_v >= VR) continue;
    if (SPLIT) {  // unnormalised partial of this key chunk: [128 virtual rows][HD], (max, sum) per row
      const long long pbase = (((long long)(G == 1 ? uniform(block_rank(st, s, vb)) : item) * sh.KV + kvh) * ns + chunk) * 128 + wave * 32 + 16 * b + n;
      float *op = part_o + pbase * HD + 4 * j;
#pragma unroll
      for (int h = 0; h < NT / 4; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) *(f32x4 *)(op + 4 * (NT * i + 4 * h)) = line[h][i];
      if (j == 0) *(float2 *)(part_ml + 2 * pbase) = float2{m[b], l[b]};
    } else {
      const int row = my_v / g, hg = my_v - row * g;
      const float inv = 1.0f / l[b];
      float *op = out + ((long long)(st.tok_off[s] + row) * sh.H + kvh * g + hg) * vhd + 4 * j;
#pragma unroll
      for (int h = 0; h < NT / 4; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (PAD && 4 * (NT * i + 4 * h + j) >= vhd) continue;  // (the width is a multiple of 4)
          *(f32x4 *)(op + 4 * (NT * i + 4 * h)) = line[h][i] * inv;
        }
    }
  }
}

template <int HD, bool SPLIT, int G, bool PAD, bool BIAS = false>
__global__ __launch_bounds__(G == 3 ? 256 : 512, G == 3 && HD == 64 && !BIAS ? 3 : 2) void prefill_mfma_kernel(const float *__restrict__ q_rot,
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
__global__ __launch_bounds__(512, 2) void prefill_turns_kernel(const float *__restrict__ q_rot,
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
  // With long key ranges, about 1024 row blocks and chunks: two blocks share a workgroup and its tiles then.
  const int ns_1024 = (int)((1024 + wgs - 1) / wgs);
  if (longest / ns_1024 >= 32) return ns_1024 < 16 ? ns_1024 : 16;
  // Otherwise what is estimated to end first, in times of a key tile: a compute unit has one workgroup at a time, which costs three tiles beside
  // its own; the launch that merges costs three and one and a half for each chunk, half of that where it has few rows (heads over 64, whose tiles take
  // longer: two, one and a quarter).
  // Us, chunks by a target of 512 workgroups | these: 32 / 8 heads of 64, 800 rows 49 | 41, 200 on 2000 46 | 37, 400 on 4000 113 | 89; heads of 128, 800 rows 86 | 73,
  // 32 / 4 heads, 512 on 4096 214 | 181; heads of 96, 777 rows 70 | 59.  Few rows, as many chunks as of many | these: 32 / 8 heads of 64, 17 on 2000 26.8 | 24.3, 40 on 2000
  // 28.4 | 26.2, 40 on 8000 48.1 | 46.2.
  double blocks = 0, tiles = 0;
  for (int s = 0; s < st.n_seqs; ++s) {
    const double n = (st.n_new[s] * (double)sh.g + 127) / 128;
    blocks += n;
    tiles += n * ((st.start_pos[s] + st.n_new[s] * 0.5) / 32 + 1);
  }
  // (heads over 64: not so many that two blocks share a workgroup, which walks through a whole range there with six roundings a tile)
  const double a_chunk = wgs < 128 ? 0.75 + 0.75 * wgs / 128 : 1.5;
  const int cap = longest / 8;  // at least eight key tiles per chunk
  int best = 1;
  double least = 0;
  for (int ns = 1; ns == 1 || (ns <= cap && ns <= 16 && (sh.hd <= 64 || wgs * ns <= 768)); ++ns) {
    const double rounds = (double)((wgs * ns + 255) / 256), one = (longest + ns - 1) / ns + 3, all = rounds * (tiles / blocks / ns + 3);
    const double ends = (one > all ? one : all) + (ns == 1 ? 0 : sh.hd <= 64 ? 3 + a_chunk * ns : 2 + 1.25 * ns);
    if (ns == 1 || ends < least) {
      least = ends;
      best = ns;
    }
  }
  return best;
}

size_t prefill_partial_floats(const Shape &sh, int items, int ns, int v_hd) {
  return ns > 1 ? (size_t)items * sh.KV * ns * 128 * (prefill_tile_head_dim(widest(sh, v_hd)) + 2) : 0;
}

// How many key tiles a row block of a sequence walks through on average (per: blocks that walk together), all chunks of them.
static double mean_tiles(const SeqTable &st, const Shape &sh, int s, int per) {
  return (st.start_pos[s] + 0.5 * st.n_new[s] + 64.0 * per / sh.g) / 32 + 0.5;
}

static long long block_pairs(const SeqTable &st) {
  long long pairs = 0;
  for (int s = 0; s < st.n_seqs; ++s) pairs += (st.work_off[s] + 1) / 2;
  return pairs;
}

PrefillLaunch plan_prefill_launch(const SeqTable &st, const Shape &sh, int items, int ns, int wgs_per_cu, int groups, int v_hd) {
  PrefillLaunch p;
  p.n_wgs = (long long)items * sh.KV * ns;
  const int tile_hd = prefill_tile_head_dim(widest(sh, v_hd));
  p.groups = groups >= 1 && groups <= 3 ? groups : 2;
  if (p.groups != groups) {
    int longest = 0;
    double tiles = 0, pair_tiles = 0, rows = 0;
    const long long pairs = block_pairs(st);
    for (int s = 0; s < st.n_seqs; ++s) {
      const int n = (st.start_pos[s] + st.n_new[s] + 31) / 32;
      longest = n > longest ? n : longest;
      tiles += st.work_off[s] * mean_tiles(st, sh, s, 1);
      pair_tiles += (st.work_off[s] + 1) / 2 * mean_tiles(st, sh, s, 2);
      rows += (double)st.n_new[s] * sh.g;
    }
    if (p.n_wgs <= 768) {
      // Up to three row blocks a compute unit: each in a workgroup of two groups that share its keys, but for ranges too short to share, which one group
      // has walked through in the time of the two groups' merge, and of which two or three share a compute unit.  Us, two groups | one: 32 / 8 heads
      // of 64, 20 rows 10.0 | 8.6, 45 rows 10.6 | 9.7, 100 rows 13.1 | 12.2, 128 rows 14.1 | 14.3, 200 rows 16.2 | 17.7; heads of 128, 45 rows 14.2 | 12.4, 64 rows
      // 16.0 | 14.8, 128 rows 19.5 | 20.3; more than 256 blocks: 16 sequences of 100 rows 24.7 | 16.5 and 40 | 24.6, 8 of 200 rows 27.4 | 22.6 and 40.6 | 33.9.
      if (ns == 1 && longest <= (p.n_wgs > 256 ? 8 : tile_hd == 64 ? 4 : 3)) p.groups = 3;
    } else {
      // More: two blocks a workgroup, which share a tile's splits and of whose groups one has MFMAs while the other has none, or a workgroup a block,
      // two or three on a compute unit, which start and end beside each other and leave no half empty where a sequence has an odd block.  What is
      // estimated to end first, in us: 256 pairs take 7 and, a key tile, 1.1 to 2.6 by how full they are (heads over 64: 12.5, 1.6 to 4.6), 256 blocks
      // 3.2 and 1.1 a tile, longer ranges 1.43 (5.5 and 2.45).
      // Us, two blocks | one: 64 sequences, 32 / 8 heads of 64, of 40 rows 25.5 | 22.2, 100 rows 59.6 | 44.3, 200 rows 135 | 96, 400 rows 330 | 282, 40 on 500 82 | 96,
      // 100 on 2000 634 | 733; one of 4096 rows 343 | 351; heads of 128, of 40 rows 39 | 36, 200 rows 228 | 198, 100 on 500 357 | 410; 32 heads of 96, of 100 rows
      // (a block each) 157 | 110, 40 on 500 397 | 320, 400 rows 671 | 700.
      const double walk = tiles / items / ns, pair_walk = pair_tiles / pairs / ns, full = rows / (256.0 * pairs);
      const double two = pairs * sh.KV * ns / 256.0 * (tile_hd == 64 ? 7 + (1.1 + 1.5 * full) * pair_walk : 12.5 + (1.6 + 3 * full) * pair_walk);
      const double one = p.n_wgs / 256.0 * (tile_hd > 64 ? 5.5 + 2.45 * walk : walk < 13 ? 3.2 + 1.1 * walk : 1.43 * walk - 1.1);
      p.groups = one < two ? 3 : 1;
    }
  }
  p.pad = 0;
  // Eight wavefronts fill a compute unit's registers.  Of the workgroups of four, up to 256 have one each to themselves, more as many as fit.
  p.wgs_per_cu = p.groups != 3 ? 1 : wgs_per_cu >= 1 && wgs_per_cu <= 3 ? wgs_per_cu : p.n_wgs <= 256 ? 1 : 0;
  if (p.groups == 3 && p.wgs_per_cu) {
    const size_t static_lds = (size_t)16 * (tile_hd == 64 ? kLdsUnits<64, 3> : kLdsUnits<128, 3>);
    const size_t want = (size_t)160 * 1024 / p.wgs_per_cu;  // one more workgroup would not fit
    const size_t floor_ = (size_t)160 * 1024 / (p.wgs_per_cu + 1) + 256;
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

long long prefill_workgroups(const SeqTable &st, const Shape &sh, const PrefillLaunch &p, int items, int ns) {
  if (p.turns) return (p.n_wgs + p.turns - 1) / p.turns;
  return (p.groups == 1 ? block_pairs(st) : items) * sh.KV * ns;
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
  const PrefillLaunch plan = plan_prefill_launch(st, sh, items, ns, wgs_per_cu, groups_wanted, v_hd);
  const long long n_wgs = plan.n_wgs;
  if (n_wgs > 0x7fffffffLL) return hipErrorInvalidValue;
  // the kernels address a row of a (sequence, kv head) by a 32-bit byte offset from its first row
  if ((long long)sh.cap * sh.hd * 4 > 0xffffffffLL) return hipErrorInvalidValue;
  const float c = scale * kLog2e;
  dim3 grid((unsigned)prefill_workgroups(st, sh, plan, items, ns));
  float *part_o = partials;
  float *part_ml = partials ? partials + (size_t)items * sh.KV * ns * 128 * tile_hd : nullptr;
  const int groups = plan.groups;
  const size_t lds_pad = plan.pad;
  if (plan.turns) {
#define SHAINET_LAUNCH_TURNS(HD_, ...)                                                                          \
  SHAINET_LAUNCH_TIMED((prefill_turns_kernel<HD_, 2, __VA_ARGS__>), grid, dim3(512), 0, stream, before, after, q_rot, kc, \
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
    if (groups == 3)                                                                                            \
      SHAINET_LAUNCH_TIMED((prefill_mfma_kernel<HD_, SPLIT_, 3, __VA_ARGS__>), grid, dim3(256), lds_pad, stream, before, \
                           main_after, q_rot, kc, vc, out, part_o, part_ml, st, sh, ns, c, db);                     \
    else if (groups == 2)                                                                                       \
      SHAINET_LAUNCH_TIMED((prefill_mfma_kernel<HD_, SPLIT_, 2, __VA_ARGS__>), grid, dim3(512), lds_pad, stream, before, \
                           main_after, q_rot, kc, vc, out, part_o, part_ml, st, sh, ns, c, db);                     \
    else                                                                                                        \
      SHAINET_LAUNCH_TIMED((prefill_mfma_kernel<HD_, SPLIT_, 1, __VA_ARGS__>), grid, dim3(512), lds_pad, stream, before, \
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
