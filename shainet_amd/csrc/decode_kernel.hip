// Split-K (flash-decoding) attention of one new row per sequence over the device
// KV cache, for gfx950.  Replaces the T = 1 case of attention_heads_cpu
// (llama_block.cr:302-401) and of the reference's attention_kv_kernel
// (cuda_kernels.cu:734-806), which launches one block per query head and walks
// the keys serially.
//
// Work split.  The key ranges of all (sequence, kv head) pairs are laid end to
// end in units of 16-key tiles and cut into equal contiguous spans, one per
// workgroup, so every workgroup streams the same number of bytes whatever the
// sequence lengths are.  Short launches (spans under 32 tiles) have their pairs rounded up to whole
// spans instead where that costs no more workgroups, so that every workgroup has one segment:
// there the second segment, not the bytes, is what a launch waits for (plan_decode).
// A span that crosses a pair boundary is processed as two segments.  The four wavefronts of a workgroup take the tiles of the span
// round-robin (across segments), each keeping its own online softmax per segment,
// and merge through LDS into one partial (max, sum, O) per segment; the workgroup
// that holds the end of a pair waits, once its own span is done, for the partials
// of the workgroups that hold the pair's earlier parts (flag words say when a
// partial is complete; the merging workgroup clears them again), merges them in a
// fixed order and writes the output row, so a decode step is one launch.  Nothing
// a workgroup does between two segments waits for another workgroup or for memory:
// a wavefront's first tile of the next segment is fetched during its last tile of
// this one, and a partial is marked complete one tile later.
//
// Per 16-key tile a wavefront
//   * copies the K tile (16 contiguous rows) from HBM straight into LDS with
//     global_load_lds_dwordx4, 1 KiB per instruction, fully coalesced, with the
//     16-byte pieces of each row XOR-swizzled so that the later ds_read_b128 of
//     MFMA operands is bank-conflict free;
//   * loads the V tile into registers (256 contiguous bytes per 16 lanes);
//   * computes S^T = K Q^T with v_mfma_f32_16x16x4_f32: rows = keys, columns =
//     the g query heads of the GQA group, so K and V are read once per group;
//   * updates the online softmax with wavefront shuffles, and accumulates
//     O^T += V^T P^T with the probabilities taken directly from the S^T
//     accumulator registers (they already have the B-operand layout).
// The loads of tile t+1 are issued before the arithmetic of tile t.
//
// MFMA 16x16x4 operand layout (lane l): A[m = l%16][k = l/16], B[k = l/16][n = l%16],
// D[m = 4*(l/16) + r][n = l%16] for accumulator register r = 0..3.  The
// contraction index may be visited in any order as long as A and B agree:
//   scores: k-step s of lane group j = l/16 covers d = 16*(s/4) + 4*j + s%4;
//   output: tile t, row m is d = 64*(t/4) + 4*m + t%4; k-step r of lane group j is
//           key 4*j + r of the tile, where accumulator register r of S^T lives.
#include "attn_kernels.hpp"
#include "lane_quarters.hpp"
#include "lds_copy.hpp"

#include <math.h>
#include <stdint.h>
#include <stdlib.h>

namespace shainet {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Split-K partials cross workgroups that may sit on different XCDs, whose L2
// caches are not kept coherent with each other for ordinary accesses.  Relaxed
// atomic accesses at agent scope compile to write-through stores and cache-
// bypassing loads, which is all that is needed for data published through a
// flag word written after them.
__device__ __forceinline__ void coherent_store(float *p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void coherent_store4(float *p, f32x4 v) {  // the same, 16 bytes at a time
  asm volatile("global_store_dwordx4 %0, %1, off sc1" : : "v"(p), "v"(v) : "memory");
}
__device__ __forceinline__ float coherent_load(const float *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

#define LDS_PTR(p) ((__attribute__((address_space(3))) void *)(uintptr_t)(p))
#define GLOBAL_PTR(p) ((const __attribute__((address_space(1))) void *)(p))

template <int HD>
struct DecodeCfg {
  static constexpr int NT = HD / 16;         // float4 of K per lane per tile; d tiles of the output
  static constexpr int PPR = HD / 4;         // 16-byte pieces per row
  static constexpr int ROW_BYTES = HD * 4;
  static constexpr int TILE_BYTES = 16 * ROW_BYTES;
  static constexpr int NKI = TILE_BYTES / 1024;  // global_load_lds instructions per K tile
  static constexpr int NVU = HD / 64;            // float4 of a V row per lane
};

// K and V rows are read once per launch and there are far more of them than the caches hold:
// they are loaded with the non-temporal hint (`nt`), which tells the caches not to keep them.
// Measured on the batch of 16 sequences of 2048 to 8192 keys: 112.2 -> 102.5 us per launch, and
// 181 -> 162 us with every sequence at 8192; the cache-scope bits on top of it change nothing.
constexpr int kNonTemporal = 2;  // the nt bit of the cache-policy operand

// PAD: the head dimension hd of the data is any multiple of 4 up to HD, the head dimension the
// tiles are laid out for.  The query's elements beyond hd are zeros, so whatever stands in for
// the keys' there does not reach the scores, and output elements beyond hd are never stored;
// the pieces of a tile beyond hd repeat the row's first piece (a cache hit, no HBM traffic).
// Without PAD hd == HD and no instruction is spent on any of this.
//
// Issue the asynchronous copy of the K tile starting at row `kb` into `lds`.
template <int HD, bool PAD>
__device__ __forceinline__ void issue_k_tile(const float *kbase, int kb, int last_row, char *lds, int lane, int hd) {
  using C = DecodeCfg<HD>;
#pragma unroll
  for (int u = 0; u < C::NKI; ++u) {
    const int slot = u * 64 + lane;
    const int row = slot / C::PPR, q = slot % C::PPR;
    int piece = q ^ row;  // row < 16 only touches the low four bits
    if (PAD) piece = 4 * piece < hd ? piece : 0;
    const float *src = kbase + (long long)min(kb + row, last_row) * (PAD ? hd : HD) + 4 * piece;
    __builtin_amdgcn_global_load_lds(GLOBAL_PTR(src), LDS_PTR(lds + u * 1024), 16, 0, kNonTemporal);
  }
}

template <int HD, bool PAD>  // hd: floats per row of V
__device__ __forceinline__ void load_v_tile(const float *vbase, int kb, int last_row, int col, int j,
                                            f32x4 (&v)[4][DecodeCfg<HD>::NVU], int hd) {
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float *vp = vbase + (long long)min(kb + 4 * j + r, last_row) * (PAD ? hd : HD);
#pragma unroll
    for (int u = 0; u < DecodeCfg<HD>::NVU; ++u) {
      int d = 4 * col + 64 * u;
      if (PAD) d = d < hd ? d : 0;
      v[r][u] = __builtin_nontemporal_load((const f32x4 *)(vp + d));
    }
  }
}

// Spans: eight consecutive workgroups share 8 * tiles_per_wg tiles of the stream, workgroup
// 8k + r taking tiles [off[r], off[r + 1]) of them (SpanTable, made by plan_decode).  Workgroups
// go to the eight XCDs round-robin by index, and the XCDs of the machines measured do not
// stream equally fast (see plan_decode), so equal spans would not end together.
__device__ __forceinline__ int span_begin(int w, int tiles_per_wg, const SpanTable &sp) {
  return (w >> 3) * 8 * tiles_per_wg + sp.off[w & 7];
}
__device__ __forceinline__ int workgroup_of_tile(int t, int tiles_per_wg, const SpanTable &sp) {
  const int k = t / (8 * tiles_per_wg), rel = t - k * 8 * tiles_per_wg;
  int r = 0;
#pragma unroll
  for (int i = 1; i < 8; ++i) r += rel >= sp.off[i] ? 1 : 0;
  return 8 * k + r;
}

// Tiles of a pair in the stream: rounded up to whole spans where spans end with the pairs (align > 1).
__host__ __device__ inline int padded_tiles(int n_s, int align) {
  return align > 1 ? (n_s + align - 1) / align * align : n_s;
}
// The kernel's way to the same: by = 2^32 / align, rounded up (0: spans do not end with the pairs), which gives the
// quotient of numbers below 2^27 exactly for divisors up to 31; a division in front of the first loads cost a short
// launch 0.3 us.
__host__ __device__ inline unsigned align_factor(int align) { return align > 1 ? 0xffffffffu / (unsigned)align + 1u : 0u; }
__device__ __forceinline__ int padded_tiles_by(int n_s, int align, unsigned by) {
  return by ? (int)(__umulhi((unsigned)(n_s + align - 1), by) * (unsigned)align) : n_s;
}

// One segment of a workgroup's span: tiles [tile0, tile1) of one (sequence, kv head) pair.
struct Segment {
  int s, kvh, R, L, n_s, tile0, tile1, token;  // R new rows; L keys visible to the last of them
  int n_p, next;  // the pair's tiles in the stream (n_s, rounded up: plan_decode); where the stream goes on behind the segment
  int rot;  // the segment's tiles are visited from tile0 + rot on, wrapping round to tile0 + rot - 1
  const float *kbase, *vbase;
};

// Where a workgroup starts within a segment.  Workgroups that all walk their spans from the first
// tile on move through memory in step, a fixed number of bytes apart, and for some distances
// (129 or 145 tiles of 8 KiB, for one) their requests pile up on a few memory channels: a plain
// read kernel laid out that way drops from 6.1 to 5.2 and 4.8 TB/s, and keeps 6.0 TB/s at every
// distance when each workgroup starts at a different place of its range.  The order of the keys
// does not matter to an online softmax.
__device__ __forceinline__ int segment_rotation(int n_tiles, unsigned rotate) {
  if (!rotate || n_tiles < 2) return 0;
  return (int)(((blockIdx.x * 2654435761u) >> 12) % min((unsigned)n_tiles, rotate));
}

// The segment that starts at tile t of the stream; s: a sequence at or before t's, moved up to it.
__device__ __forceinline__ Segment segment_at(int t, int t_end, int &s, const SeqTable &st, const Shape &sh, int hd,
                                              int vhd, bool own_v_rows, const float *kc, const float *vc, unsigned rotate,
                                              int align, unsigned align_by) {
  while (s + 1 < st.n_seqs && t >= st.work_off[s + 1]) ++s;
  Segment g;
  g.s = s;
  g.R = st.n_new[s];
  g.L = st.start_pos[s] + g.R;  // visible keys of the last new row
  g.n_s = (g.L + 15) >> 4;    // tiles per kv head of this sequence
  g.n_p = padded_tiles_by(g.n_s, align, align_by);
  const int rel = t - st.work_off[s];
  g.kvh = rel / g.n_p;
  g.tile0 = rel - g.kvh * g.n_p;
  g.next = min(t + g.n_p - g.tile0, t_end);
  g.tile1 = min(g.n_s, g.tile0 + (g.next - t));  // (never empty: a span starts in front of the pair's last tile)
  g.rot = __builtin_amdgcn_readfirstlane(segment_rotation(g.tile1 - g.tile0, rotate));
  const long long head_base = (long long)st.slot[s] * sh.seq_stride + (long long)g.kvh * sh.cap * hd;
  g.kbase = kc + head_base;
  g.vbase = vc + (own_v_rows ? ((long long)st.slot[s] * sh.KV + g.kvh) * sh.cap * vhd : head_base);
  g.token = st.tok_off[s];
  return g;
}

constexpr int kFlagSpinLimit = 1 << 21;  // polls of about a microsecond each: seconds

// part_flag: NW words per partial slot, zero between launches: each wavefront sets its word of
// a partial once its share is in memory, the workgroup that merges the pair clears the words it waited for
// (so a launch may be replayed as it is).  error: set when the wait for other workgroups'
// partials was given up, after spin_limit polls.  flag_set: where the marks are written; the
// same as part_flag except in the test of that give-up, which sends them elsewhere.
// DEV: the sequence table and the spans come from *dev (device memory, written by
// decode_plan_kernel earlier on the stream) instead of from the kernel arguments.
struct ReadAhead {
  const float *w;  // [2 n, k]
  int k, n, first_wg;
};

// Workgroup ah.first_wg + j reads the rows 4 j .. 4 j + 3 and n + the same of ah.w and drops them.
__device__ __forceinline__ void read_ahead(const ReadAhead &ah) {
  const int row = 4 * ((int)blockIdx.x - ah.first_wg) + (int)(threadIdx.x >> 6);
  if (row >= ah.n) return;
  const int pieces = ah.k >> 8;  // 16-byte pieces per lane and row
  for (int half = 0; half < 2; ++half) {
    const float *p = ah.w + ((long long)half * ah.n + row) * ah.k + 4 * (threadIdx.x & 63);
    for (int i0 = 0; i0 < pieces; i0 += 8) {
      f32x4 v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = *(const f32x4 *)(p + 256 * min(i0 + u, pieces - 1));
#pragma unroll
      for (int u = 0; u < 8; ++u) asm volatile("" : : "v"(v[u]));
    }
  }
}

// The arithmetic of norm_rotate_pair (prep_math.hpp) in the layouts of the kernel below, the same bits: no product fuses
// into an add.
#pragma clang fp contract(off)
__device__ __forceinline__ void norm_rotate_quad(f32x4 &x0, f32x4 &x1, bool has_w, f32x4 w0, f32x4 w1, float inv, f32x4 cs01,
                                                 f32x4 cs23) {
#pragma clang fp contract(off)
  const f32x4 c = {cs01.x, cs01.z, cs23.x, cs23.z}, s = {cs01.y, cs01.w, cs23.y, cs23.w};
  if (has_w) {
    x0 = x0 * inv;
    x0 = x0 * w0;
    x1 = x1 * inv;
    x1 = x1 * w1;
  }
  const f32x4 p0 = x0 * c, p1 = x1 * s, p2 = x1 * c, p3 = x0 * s;
  x0 = p0 - p1;
  x1 = p2 + p3;
}

// 1 / rms of up to 32 head rows, the squares of a row added up one after the other as the reference does: lane r walks
// the first half of row r, lane 32 + r goes on with the second.
template <int HD>
struct SquareSum {
  f32x4 x[HD / 8];
  __device__ __forceinline__ void request(const float *row, int lane) {  // row: lane % 32's
#pragma unroll
    for (int i = 0; i < HD / 8; ++i) x[i] = *(const f32x4 *)(row + (lane >> 5) * (HD / 2) + 4 * i);
  }
  __device__ __forceinline__ float add_up(float ss) const {
#pragma clang fp contract(off)
#pragma unroll
    for (int i = 0; i < HD / 8; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float sq = x[i][e] * x[i][e];
        ss = ss + sq;
      }
    return ss;
  }
  __device__ __forceinline__ float factor(double eps, int lane) const {  // in lanes 32 + r
    const float first = add_up(0.0f);
    const float mean = add_up(__shfl(first, lane & 31)) / (float)HD;
    return (float)(1.0 / sqrt((double)mean + eps));
  }
};

// Queries as the score MFMAs take them: lane group j holds elements 16 i + 4 j .. + 3 of a head, and so both halves
// of its pairs.
template <int HD>
struct PreparedQueries {
  static constexpr int NT = HD / 16;
  f32x4 x[NT], w[NT], cs[NT];
  __device__ __forceinline__ void request(const float *row, const float *norm, const float2 *table, int j) {
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      x[i] = *(const f32x4 *)(row + 16 * i + 4 * j);
      w[i] = norm ? *(const f32x4 *)(norm + 16 * i + 4 * j) : f32x4{1.f, 1.f, 1.f, 1.f};
      cs[i] = *(const f32x4 *)(table + 16 * (i / 2) + 4 * j + 2 * (i % 2));
    }
  }
  __device__ __forceinline__ void finish(bool has_w, float inv, float (&q)[HD / 4]) {
#pragma unroll
    for (int i = 0; i < NT / 2; ++i) {
      norm_rotate_quad(x[i], x[i + NT / 2], has_w, w[i], w[i + NT / 2], inv, cs[2 * i], cs[2 * i + 1]);
#pragma unroll
      for (int e = 0; e < 4; ++e) q[4 * i + e] = x[i][e], q[4 * (i + NT / 2) + e] = x[i + NT / 2][e];
    }
  }
};

// The new key and value row of a pair, in one wavefront: lane l holds elements 4 l .. + 3 and HD / 2 + 4 l .. + 3 of the
// key (l < HD / 8, the others as lane l % (HD / 8)), and 4 (l % 16) .. + 3 of every 64 of the value.
template <int HD>
struct NewRow {
  static constexpr int kLanes = HD / 8;
  f32x4 key[2], w[2], cs[2], value[HD / 64];
  __device__ __forceinline__ void request(const float *k, const float *v, const float *norm, const float2 *table, int lane) {
    const int e = 4 * (lane % kLanes);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      key[h] = *(const f32x4 *)(k + h * (HD / 2) + e);
      w[h] = norm ? *(const f32x4 *)(norm + h * (HD / 2) + e) : f32x4{1.f, 1.f, 1.f, 1.f};
      cs[h] = *(const f32x4 *)(table + e + 2 * h);
    }
#pragma unroll
    for (int u = 0; u < HD / 64; ++u) value[u] = *(const f32x4 *)(v + 64 * u + 4 * (lane & 15));
  }
  __device__ __forceinline__ void finish(bool has_w, float inv) { norm_rotate_quad(key[0], key[1], has_w, w[0], w[1], inv, cs[0], cs[1]); }
  // into row `row` of a K tile in LDS
  __device__ __forceinline__ void put_key(char *tile, int row, int lane) const {
    if (lane >= kLanes) return;
#pragma unroll
    for (int h = 0; h < 2; ++h) *(f32x4 *)(tile + row * (HD * 4) + (((lane + h * kLanes) ^ row) << 4)) = key[h];
  }
  __device__ __forceinline__ void append(float *k, float *v, int lane) const {
    if (lane < kLanes) {
      *(f32x4 *)(k + 4 * lane) = key[0];
      *(f32x4 *)(k + HD / 2 + 4 * lane) = key[1];
    }
#pragma unroll
    for (int u = 0; u < HD / 64; ++u)
      if (lane < 16) *(f32x4 *)(v + 64 * u + 4 * lane) = value[u];
  }
};
#pragma clang fp contract(fast)

// AHEAD: workgroups from ah.first_wg on (a multiple of 8) do not attend: workgroup first_wg + j
// reads the rows 4 j .. 4 j + 3 and n + the same of ah.w with ordinary loads and drops them, so
// that the launch that needs them next finds them in its XCD's L2 (a decode step of one sequence
// leaves the memory system idle while it waits on its chain of dependent loads).
// PREP: q, k and v are a projection's rows, one new row per sequence, and every workgroup has one segment
// (DecodePlan::align): each wavefront norms and rotates the queries of its group for itself, the one that holds the
// pair's last tile does the same for the new key, puts it and the new value in the place of the tile's rows
// from L - 1 on, which are not in memory yet, and appends them behind its last tile.  The launch in front that did all
// this, and the wait between the two, are gone: one sequence of 1024 positions, 8 kv heads of 64, 10.8 -> 6.7 us a call; a
// step of a QK-normed model of width 1024 3 us shorter per layer.  The sums of squares are a chain of hd additions (0.2
// to 0.5 us), which the first tile's way hides.
// BIAS (with PAD): scores gain a value by distance (DistanceBias), value rows have a width of their own.
template <int HD, int NW, bool DEV, bool PAD, bool AHEAD = false, bool BIAS = false, bool PREP = false>
__global__ __launch_bounds__(64 * NW, NW == 4 && HD <= 128 ? 2 : 1) void decode_splitk_kernel(
    const float *__restrict__ q_rot, const float *__restrict__ kc, const float *__restrict__ vc,
    float *__restrict__ out, float *part_o, float *part_ml, unsigned *part_flag, unsigned *flag_set,
    int spin_limit, int *error, SeqTable st_arg, Shape sh, int tiles_per_wg_arg, SpanTable sp_arg, int total_tiles_arg,
    int align_arg, unsigned align_by_arg, int n_slots, int pstride, float c, unsigned rotate, const DecodeDevicePlan *__restrict__ dev, ReadAhead ah,
    DistanceBias db, PrepArgs raw) {
  static_assert(PAD || !BIAS, "sizes of their own come with padding");
  static_assert(!PREP || (!PAD && !DEV && HD <= 128), "preparation of plain host-planned rows");
  if constexpr (AHEAD) {
    if ((int)blockIdx.x >= ah.first_wg) {
      read_ahead(ah);
      return;
    }
  }
  using C = DecodeCfg<HD>;
  const SeqTable &st = DEV ? dev->st : st_arg;
  const SpanTable &sp = DEV ? dev->spans : sp_arg;
  const int tiles_per_wg = DEV ? dev->tiles_per_wg : tiles_per_wg_arg;
  const int total_tiles = DEV ? dev->total_tiles : total_tiles_arg;
  const int align = DEV ? dev->align : align_arg;
  const unsigned align_by = DEV ? dev->align_by : align_by_arg;
  constexpr int NT = C::NT;
  // per wavefront two K tile buffers; after a segment's last tile the wavefront parks its O
  // rows [g][HD] in one while the other already receives the next segment's first tile
  __shared__ __attribute__((aligned(1024))) char k_lds[NW][2][C::TILE_BYTES];
  __shared__ float sm_m[NW][16], sm_l[NW][16];  // per wavefront and head: running max, sum
  __shared__ int sm_park[NW];                   // where each wavefront parked its O rows
  constexpr int TILE_FLOATS = C::TILE_BYTES / 4;
  constexpr int WAVE_LDS_FLOATS = 2 * TILE_FLOATS;  // floats between two wavefronts' areas

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: tile numbers stay in scalar registers
  const int col = lane & 15, j = lane >> 4;
  const int g = sh.g;
  const int hd = PAD ? sh.hd : HD;  // floats between two rows of q, K, V and the output
  const int vhd = BIAS ? db.v_hd : hd;  // of V and the output
  const float ce = BIAS ? 1.f : c;      // scores with a bias are kept in log2 units
  const int t_begin = span_begin(blockIdx.x, tiles_per_wg, sp);
  const int t_end = min(total_tiles, span_begin(blockIdx.x + 1, tiles_per_wg, sp));
  if (t_begin >= t_end) return;  // unequal spans can leave the last workgroup without tiles
  char *my_lds = &k_lds[wave][0][0];

  int t = t_begin;
  // The sequence the span starts in: every lane looks at one entry of the prefix sums (a walk
  // along them with dependent scalar loads took 2.5 us for a workgroup in the middle of 16
  // sequences).
  int s = (int)__popcll(__ballot(lane + 1 < st.n_seqs && t_begin >= st.work_off[lane + 1 < kMaxSeqs ? lane + 1 : kMaxSeqs]));
  Segment seg = segment_at(t, t_end, s, st, sh, hd, vhd, BIAS, kc, vc, rotate, align, align_by);

  f32x4 v_next[4][C::NVU];
  float qr[HD / 4];
  // columns beyond the last repeat column 0: their results are never stored, and leaving the
  // loaded values untouched here keeps the wait for them out of this place
  // MFMA column c of a segment is new row c / g, head c % g of the group (R * g <= 16 columns)
  auto load_q = [&](const Segment &sg) {
    const int cq = col < sg.R * g ? col : 0, row = cq / g;
    const int head = sg.kvh * g + (cq - row * g);
    const float *qp = q_rot + (BIAS ? (sg.token + row) * db.q_stride + (long long)head * hd : ((long long)(sg.token + row) * sh.H + head) * hd) + 4 * j;
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      f32x4 x = {0.f, 0.f, 0.f, 0.f};
      if (!PAD || 16 * i + 4 * j < hd) x = *(const f32x4 *)(qp + 16 * i);
      qr[4 * i + 0] = x.x;
      qr[4 * i + 1] = x.y;
      qr[4 * i + 2] = x.z;
      qr[4 * i + 3] = x.w;
    }
  };
  // `par`: the one of this wavefront's two buffers that holds (or is receiving) its next K tile.
  // A segment's first tile is fetched while the segment before it is still being worked on.
  int par = 0;
  // The tiles of the span go to the wavefronts round-robin as one sequence, whatever segments
  // they fall into (a fresh start per segment would leave one wavefront with a tile more than
  // its share in every segment): this wavefront's first place in the visiting order of the
  // segment at stream position ts, and the tile at place i of that order.
  auto first_place = [&](int ts) { return (wave - (ts - t_begin)) & (NW - 1); };
  auto tile_at = [&](const Segment &sg, int i) {
    const int n = sg.tile1 - sg.tile0, k = i + sg.rot;
    return sg.tile0 + (k < n ? k : k - n);
  };
  static_assert((NW & (NW - 1)) == 0, "round-robin by masking");
  // start fetching the tile at key row `row` into buffer `which`
  auto fetch = [&](int which, const float *kb_, const float *vb_, int row, int last_row) {
    issue_k_tile<HD, PAD>(kb_, row, last_row, my_lds + which * C::TILE_BYTES, lane, hd);
    load_v_tile<HD, PAD>(vb_, row, last_row, col, j, v_next, vhd);
  };
  // PREP: the last row in memory
  auto last_row = [&](const Segment &sg) { return PREP ? max(sg.L - 2, 0) : sg.L - 1; };
  NewRow<HD> fresh;
  bool holds_new = false;  // this wavefront has the pair's last tile
  if constexpr (PREP) {
    // (all of it is requested in front of the first tile, and arrives in front of it)
    const int n = seg.tile1 - seg.tile0, last = seg.n_s - 1 - seg.tile0 - seg.rot;
    holds_new = seg.tile1 == seg.n_s && ((last < 0 ? last + n : last) & (NW - 1)) == wave;
    const float *qrow = raw.q + seg.token * raw.q_stride + (long long)seg.kvh * g * HD;
    const float *krow = raw.k + seg.token * raw.k_stride + (long long)seg.kvh * HD;
    const float2 *cs = raw.rope_tab + (long long)(seg.L - 1) * (HD / 2);
    PreparedQueries<HD> pq;
    pq.request(qrow + (col < g ? col : 0) * HD, raw.q_norm, cs, j);
    if (holds_new) fresh.request(krow, raw.v + seg.token * raw.v_stride + (long long)seg.kvh * HD, raw.k_norm, cs, lane);
    float inv = 1.f;
    if (raw.q_norm || raw.k_norm) {  // row r: head r of the group; row g: the new key
      const int r = lane & 31;
      SquareSum<HD> sum;
      sum.request(r == g ? krow : qrow + (r < g ? r : 0) * HD, lane);
      if (first_place(t) < n) fetch(0, seg.kbase, seg.vbase, tile_at(seg, first_place(t)) * 16, last_row(seg));
      inv = sum.factor(raw.eps, lane);
    } else if (first_place(t) < n) {
      fetch(0, seg.kbase, seg.vbase, tile_at(seg, first_place(t)) * 16, last_row(seg));
    }
    pq.finish(raw.q_norm != nullptr, __shfl(inv, 32 + (col < g ? col : 0)), qr);
    if (holds_new) fresh.finish(raw.k_norm != nullptr, __shfl(inv, 32 + g));
  } else {
    if (first_place(t) < seg.tile1 - seg.tile0) fetch(0, seg.kbase, seg.vbase, tile_at(seg, first_place(t)) * 16, seg.L - 1);
    load_q(seg);
  }

  // the pair whose last segment this workgroup holds without holding all of it: merged at the
  // end of the span (only a span's first segment can start inside a pair, so there is one at most)
  bool have_merge = false;
  Segment mseg = seg;
  // this wavefront's share of a partial is written but not yet marked complete (slot, or -1):
  // the mark follows the next wait for loads, which then also covers those stores
  int pending = -1;
  auto mark_pending = [&]() {
    if (pending >= 0) {
      if (lane == 0)
        __hip_atomic_store(&flag_set[NW * pending + wave], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      pending = -1;
    }
  };

  for (;;) {
    const int L = seg.L, tile1 = seg.tile1;
    const float *kbase = seg.kbase, *vbase = seg.vbase;
    const int nc = seg.R * g;                                   // columns in use
    const int Lc = L - (seg.R - 1 - (col < nc ? col : 0) / g);  // keys visible to this lane's column
    // entry of key row k: bias_row[k]
    const float *bias_row = nullptr;
    if constexpr (BIAS) {
      const int cq = col < nc ? col : 0;
      bias_row = db.tab + (long long)(seg.kvh * g + cq % g) * db.stride + (db.origin - (Lc - 1));
    }
    // the segment after this one, if the span has one
    const int t_next = seg.next;
    const bool more = t_next < t_end;
    Segment nseg = seg;
    if (more) nseg = segment_at(t_next, t_end, s, st, sh, hd, vhd, BIAS, kc, vc, rotate, align, align_by);
    const int nplace = first_place(t_next);
    const bool nhave = more && nplace < nseg.tile1 - nseg.tile0;
    const int ntile = nhave ? tile_at(nseg, nplace) : 0;
    const int n_here = tile1 - seg.tile0;

    float m = -INFINITY, l = 0.f;
    f32x4 o[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};

    int place = first_place(t);
    // no tile of this segment for this wavefront: on to the next one's
    if (place >= n_here && nhave) fetch(par, nseg.kbase, nseg.vbase, ntile * 16, nseg.L - 1);
    for (; place < n_here; place += NW) {
      const int kb = tile_at(seg, place) * 16;
      const char *buf = my_lds + par * C::TILE_BYTES;
      par ^= 1;
      // everything issued so far (this tile's K copy and V loads) has landed:
      // s_waitcnt vmcnt(0) (expcnt and lgkmcnt fields left at their maxima), then a
      // compiler barrier so that no LDS read of the tile is scheduled above it
      __builtin_amdgcn_s_waitcnt(0x0F70);
      asm volatile("" ::: "memory");
      mark_pending();
      f32x4 v_cur[4][C::NVU];
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int u = 0; u < C::NVU; ++u) v_cur[r][u] = v_next[r][u];
      if (PREP && kb + 16 >= L) {  // the pair's last tile: nobody's key L - 1 and no value from there on is in memory
        fresh.put_key((char *)buf, L - 1 - kb, lane);
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int u = 0; u < C::NVU; ++u) v_cur[r][u] = kb + 4 * j + r >= L - 1 ? fresh.value[u] : v_cur[r][u];
        asm volatile("" ::: "memory");
      }
      // a tile that lies `reach` or more behind every column's row has no values by distance
      f32x4 near_bias = {0.f, 0.f, 0.f, 0.f};
      if constexpr (BIAS) {
        struct __attribute__((packed, aligned(4))) Four { f32x4 v; };
        if (L - seg.R - (kb + 15) < db.reach) near_bias = ((const Four *)(bias_row + kb + 4 * j))->v;
      }
      if (place + NW < n_here)
        fetch(par, kbase, vbase, tile_at(seg, place + NW) * 16, last_row(seg));
      else if (nhave)
        fetch(par, nseg.kbase, nseg.vbase, ntile * 16, nseg.L - 1);

      f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
      const char *krow = buf + col * C::ROW_BYTES;
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        const f32x4 kk = *(const f32x4 *)(krow + (((4 * i + j) ^ col) << 4));
        s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kk.x, qr[4 * i + 0], s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kk.y, qr[4 * i + 1], s1, 0, 0, 0);
        s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kk.z, qr[4 * i + 2], s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kk.w, qr[4 * i + 3], s1, 0, 0, 0);
      }
      float sv[4];
#pragma unroll
      for (int r = 0; r < 4; ++r)
        sv[r] = (kb + 4 * j + r < Lc) ? (BIAS ? (s0[r] + s1[r]) * c + near_bias[r] : s0[r] + s1[r]) : -INFINITY;
      float mx = fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3]));
      mx = fmaxf(mx, __shfl_xor(mx, 16));
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      const float mnew = fmaxf(m, mx);
      // with several new rows a column may not see any key of a late tile (-inf so far: 0 stands in)
      const float mref = mnew == -INFINITY ? 0.f : mnew;
      const float alpha = fast_exp2((m - mref) * ce);
      float p[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) p[r] = fast_exp2((sv[r] - mref) * ce);
      l = l * alpha + ((p[0] + p[1]) + (p[2] + p[3]));
      m = mnew;
#pragma unroll
      for (int i = 0; i < NT; ++i) o[i] *= alpha;
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int u = 0; u < C::NVU; ++u) {
          o[4 * u + 0] = __builtin_amdgcn_mfma_f32_16x16x4f32(v_cur[r][u].x, p[r], o[4 * u + 0], 0, 0, 0);
          o[4 * u + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(v_cur[r][u].y, p[r], o[4 * u + 1], 0, 0, 0);
          o[4 * u + 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(v_cur[r][u].z, p[r], o[4 * u + 2], 0, 0, 0);
          o[4 * u + 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(v_cur[r][u].w, p[r], o[4 * u + 3], 0, 0, 0);
        }
    }
    // the next segment's query rows (this one's are not needed any more)
    if (!PREP && more) load_q(nseg);
    if constexpr (PREP) {  // (behind the last tile: a wait for loads waits for stores, too)
      if (holds_new) {
        const long long at = (long long)(L - 1) * HD;
        fresh.append(const_cast<float *>(kbase) + at, const_cast<float *>(vbase) + at, lane);
      }
      if (seg.tile0 == 0 && wave == 0 && col < g) {
        float *qp = raw.q_rot + ((long long)seg.token * sh.H + seg.kvh * g + col) * HD + 4 * j;
#pragma unroll
        for (int i = 0; i < NT; ++i) *(f32x4 *)(qp + 16 * i) = f32x4{qr[4 * i], qr[4 * i + 1], qr[4 * i + 2], qr[4 * i + 3]};
      }
    }

    // merge the wavefronts through LDS: the wavefront parks its O rows [g][HD] in the one of
    // its two buffers that does not hold (or receive) its next tile
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    float *sm_o = (float *)&k_lds[0][0][0];
    if (col < nc) {
      float *dst = sm_o + wave * WAVE_LDS_FLOATS + (par ^ 1) * TILE_FLOATS + col * HD;
#pragma unroll
      for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) dst[64 * (i >> 2) + 4 * (4 * j + r) + (i & 3)] = o[i][r];
      if (j == 0) {
        sm_m[wave][col] = m;
        sm_l[wave][col] = l;
      }
    }
    if (lane == 0) sm_park[wave] = (par ^ 1) * TILE_FLOATS;
    // a share of an earlier partial that is still unmarked (a wavefront that had no tile since)
    if (pending >= 0) {
      __builtin_amdgcn_s_waitcnt(0x0F70);
      mark_pending();
    }
    __syncthreads();
    const bool whole_pair = seg.tile0 == 0 && tile1 == seg.n_s;
    const int pair = seg.s * sh.KV + seg.kvh;
    const int slot = blockIdx.x + pair;  // unique: both terms only grow along the tile stream
    int park[NW];
#pragma unroll
    for (int w = 0; w < NW; ++w) park[w] = w * WAVE_LDS_FLOATS + sm_park[w];
    for (int idx = threadIdx.x; idx < nc * HD; idx += 64 * NW) {
      const int cc = idx / HD, d = idx - cc * HD;
      float mm = sm_m[0][cc];
#pragma unroll
      for (int w = 1; w < NW; ++w) mm = fmaxf(mm, sm_m[w][cc]);
      const float mref = mm == -INFINITY ? 0.f : mm;  // no key of the segment visible to this column
      float acc = 0.f, ls = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const float f = fast_exp2((sm_m[w][cc] - mref) * ce);  // 0 for a wavefront that saw no visible key
        acc += f * sm_o[park[w] + cc * HD + d];
        ls += f * sm_l[w][cc];
      }
      if (whole_pair) {
        const int row = cc / g;
        if (!PAD || d < vhd) out[((long long)(seg.token + row) * sh.H + seg.kvh * g + (cc - row * g)) * vhd + d] = acc / ls;
      } else if (slot < n_slots) {
        const long long pi = (long long)slot * pstride + cc;
        coherent_store(&part_o[pi * HD + d], acc);
        if (d == 0) {
          coherent_store(&part_ml[2 * pi], mm);
          coherent_store(&part_ml[2 * pi + 1], ls);
        }
      }
    }
    const bool pair_end = !whole_pair && tile1 == seg.n_s;
    if (pair_end) {
      have_merge = true;
      mseg = seg;
    }
    // Partials are written through to device-coherent memory (coherent_store).  Each
    // wavefront marks its share complete in a word of its own once its stores are
    // acknowledged, which the next wait for a tile tells (the barrier alone does not).
    // The partial of a pair's end is read by this workgroup only.
    if (!whole_pair && !pair_end && slot < n_slots) pending = slot;
    // the parked rows are read: the next tiles may land there (with a copy into LDS in flight
    // the barriers here also wait for this wavefront's loads: the compiler's rule, which is
    // what a boundary inside a span still costs)
    __syncthreads();
    if (!more) break;
    seg = nseg;
    t = t_next;
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // this wavefront's last stores are acknowledged
  mark_pending();

  if (have_merge) {
    // This workgroup holds the end of a pair that others began: they have lower indices, were
    // started before this one and wait for nobody, so waiting for their partials is safe.
    const int a = st.work_off[mseg.s] + mseg.kvh * mseg.n_p;  // the pair's tiles are [a, a + n_s)
    const int w_lo = workgroup_of_tile(a, tiles_per_wg, sp);
    const int n_part = (int)blockIdx.x - w_lo + 1;
    const int pair = mseg.s * sh.KV + mseg.kvh;
    if (wave == 0) {
      // NW words per partial; the last of the n_part partials is this workgroup's own
      unsigned *fl = part_flag + NW * (w_lo + pair);
      for (int spins = 0;; ++spins) {
        bool ok = true;
        for (int i = lane; i < NW * (n_part - 1); i += 64)
          ok = ok && __hip_atomic_load(fl + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u;
        if (__all(ok)) {
          for (int i = lane; i < NW * (n_part - 1); i += 64)
            __hip_atomic_store(fl + i, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          break;
        }
        if (spins >= spin_limit) {
          if (lane == 0) *error = 1;
          break;
        }
        __builtin_amdgcn_s_sleep(2);
      }
    }
    __syncthreads();
    // every partial of the pair is in memory: drop whatever this XCD's caches
    // still hold of those addresses, then read them with ordinary wide loads
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    constexpr int LPR = HD / 4;       // lanes that cover one row with float4
    constexpr int GROUPS = 64 / LPR;  // partials handled side by side
    const int d4 = lane % LPR, grp = lane / LPR;
    const long long base = (long long)(w_lo + pair) * pstride;  // partial of workgroup w, column cc: base + (w - w_lo) * pstride + cc
    for (int cc = wave; cc < mseg.R * g; cc += NW) {
      const long long first = base + cc;
      // the largest of the partials' maxima: from a pass of its own over them, or, when one
      // round of loads covers all partials, from that round (one memory round trip less)
      const bool one_round = n_part <= 8 * GROUPS;
      float mm = -INFINITY;
      if (!one_round) {
        for (int i = lane; i < n_part; i += 64) mm = fmaxf(mm, part_ml[2 * (first + (long long)i * pstride)]);
        for (int o2 = 32; o2 > 0; o2 >>= 1) mm = fmaxf(mm, __shfl_xor(mm, o2));
      }
      float ls = 0.f;
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
      for (int i0 = 0; i0 < n_part; i0 += 8 * GROUPS) {  // eight rows in flight per lane
        f32x4 x[8];
        float f[8], lp[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int i = i0 + u * GROUPS + grp;
          const long long pi = first + (long long)min(i, n_part - 1) * pstride;
          x[u] = *(const f32x4 *)&part_o[pi * HD + 4 * d4];
          f[u] = part_ml[2 * pi];
          lp[u] = part_ml[2 * pi + 1];
        }
        if (one_round) {
#pragma unroll
          for (int u = 0; u < 8; ++u)
            if (u * GROUPS + grp < n_part) mm = fmaxf(mm, f[u]);
#pragma unroll
          for (int o2 = LPR; o2 < 64; o2 <<= 1) mm = fmaxf(mm, __shfl_xor(mm, o2));  // over the lanes of one d4
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int i = i0 + u * GROUPS + grp;
          const float w = i < n_part ? fast_exp2((f[u] - mm) * ce) : 0.f;
          acc += w * x[u];
          ls += w * lp[u];
        }
      }
#pragma unroll
      for (int o2 = LPR; o2 < 64; o2 <<= 1) {
        acc.x += __shfl_xor(acc.x, o2);
        acc.y += __shfl_xor(acc.y, o2);
        acc.z += __shfl_xor(acc.z, o2);
        acc.w += __shfl_xor(acc.w, o2);
        ls += __shfl_xor(ls, o2);
      }
      if (grp == 0 && (!PAD || 4 * d4 < vhd)) {
        const float inv = 1.0f / ls;
        const int row = cc / g;
        *(f32x4 *)&out[((long long)(mseg.token + row) * sh.H + mseg.kvh * g + (cc - row * g)) * vhd + 4 * d4] = acc * inv;
      }
    }
  }
}

// Pairs of up to 12 tiles (heads of 128: 8), a workgroup each, one new row per sequence: the arithmetic of the kernel above in its order, the
// same bits, with everything requested at once.  T: tiles per wavefront, those of the longest pair; a wavefront without a T-th one
// requests its pair's last again, so that no load hangs on a condition.  The queries (and the new key and value) are made once, in pieces of
// a few threads, and read from LDS: by every wavefront for itself, as above, they were 25 of a wavefront's 33 loads, and a compute unit takes 16
// cycles for each.  K goes to LDS by instructions that the compiler does not count: those it knows have it wait for everything in flight in front
// of any exchange between lanes.  Grid: kv heads (and workgroups that read ahead), sequences.
// Us of the launch, the kernel above | this, one sequence, 8 kv heads of 64: 61 keys 6.3 | 4.3, 125 7.2 | 5.2, 171 7.9 | 6.3; with QK-norm 31 keys
// 6.8 | 4.7, 81 7.6 | 5.7, 171 8.4 | 6.8; heads of 128, 101 keys 9.8 | 7.2, with QK-norm 11.4 | 7.8; 16 sequences of 101 keys 8.0 | 5.6, of 181 9.2 | 7.1, of
// heads of 128 with QK-norm 12.4 | 8.9.  (Every wavefront its queries, K straight to registers 5.2, 6.6, 7.8; by LDS 5.2, 6.4, 7.3.)  What bounds it, in cycles
// of 6400 for 61 keys: arguments 1200, loads requested and there 1700, queries 500, a tile's MFMAs and softmax 1900, merge and stores 1500.
struct RowSeqs {
  int start[kMaxSeqs], slot[kMaxSeqs];
};
constexpr int kRowsPlain = 0, kRowsPrep = 1, kRowsBias = 2;  // queries and new rows are prepared; are a projection's; scores gain a value by distance
template <int HD>
constexpr int kRowTiles = HD == 64 ? 3 : 2;

template <int HD, int T, int MODE>
__global__ __launch_bounds__(256, 1) void decode_rows_kernel(const float *__restrict__ q_rot, const float *__restrict__ kc,
                                                             const float *__restrict__ vc, float *__restrict__ out, const RowSeqs seqs,
                                                             Shape sh, float c, unsigned rotate, ReadAhead ah, DistanceBias db, PrepArgs raw) {
  using C = DecodeCfg<HD>;
  constexpr int NT = C::NT, NW = 4;
  constexpr bool PREP = MODE == kRowsPrep, BIAS = MODE == kRowsBias;
  const int kvh = blockIdx.x, s = blockIdx.y;
  const int start = seqs.start[s], seq_slot = seqs.slot[s];
  // (all arguments together, or those behind a condition are asked for behind it, a round trip later)
  asm volatile("" : : "s"(start), "s"(seq_slot), "s"(kc), "s"(vc), "s"(out), "s"(sh.KV), "s"(sh.g), "s"(sh.cap), "s"(sh.seq_stride), "s"(rotate));
  if constexpr (PREP)
    asm volatile("" : : "s"(raw.q), "s"(raw.k), "s"(raw.v), "s"(raw.q_stride), "s"(raw.k_stride), "s"(raw.v_stride), "s"(raw.q_norm), "s"(raw.k_norm),
                 "s"(raw.rope_tab), "s"(raw.q_rot));
  if (ah.w && kvh >= ah.first_wg) {
    read_ahead(ah);
    return;
  }
  if (kvh >= sh.KV) return;  // (between the last pair and the first that reads ahead)
  constexpr int kRow = HD + 4;  // floats from a query to the next in LDS
  __shared__ __attribute__((aligned(1024))) char k_lds[NW][T][C::TILE_BYTES];
  __shared__ __attribute__((aligned(16))) float sm_o[NW][16 * HD], sm_q[17 * kRow], sm_v[HD];
  __shared__ float sm_m[NW][16], sm_l[NW][16];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, j = lane >> 4;
  const int g = sh.g;
  const int L = start + 1, n = (L + 15) >> 4;
  const long long head_base = (long long)seq_slot * sh.seq_stride + (long long)kvh * sh.cap * HD;
  const float *kbase = kc + head_base;
  const float *vbase = vc + (BIAS ? ((long long)seq_slot * sh.KV + kvh) * sh.cap * HD : head_base);
  const float ce = BIAS ? 1.f : c;
  const int cq = col < g ? col : 0;  // columns beyond the last repeat column 0: their results are never stored

  // a thread's piece of the queries, and of the new key (row g): four elements and, to prepare, the four a half further
  constexpr int kPieces = PREP ? HD / 8 : HD / 4, kRounds = (17 * kPieces + 255) / 256;
  const int items = (PREP ? g + 1 : g) * kPieces;
  const float *qrow = PREP ? raw.q + s * raw.q_stride + (long long)kvh * g * HD
                           : q_rot + (BIAS ? s * db.q_stride + (long long)kvh * g * HD : ((long long)s * sh.H + kvh * g) * HD);
  const float *krow = PREP ? raw.k + s * raw.k_stride + (long long)kvh * HD : nullptr;
  f32x4 x[kRounds][2], w[kRounds][2], cs[kRounds][2], fresh;
  SquareSum<HD> sum;
  const bool norms = PREP && (raw.q_norm || raw.k_norm), has_items = 64 * wave < items;
  const int vi = (int)threadIdx.x - (256 - HD / 4);  // the last threads: the new value
#pragma unroll
  for (int u = 0; u < kRounds; ++u) {
    const int at = threadIdx.x + 256 * u, row = at / kPieces, e = 4 * (at % kPieces);
    if (at < items) {
      const float *src = PREP && row == g ? krow : qrow + row * HD;
      x[u][0] = *(const f32x4 *)(src + e);
      if constexpr (PREP) {
        const float *norm = row == g ? raw.k_norm : raw.q_norm;
        const float2 *table = raw.rope_tab + (long long)(L - 1) * (HD / 2) + e;
        x[u][1] = *(const f32x4 *)(src + HD / 2 + e);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          w[u][h] = f32x4{1.f, 1.f, 1.f, 1.f};
          if (norm) w[u][h] = *(const f32x4 *)(norm + h * (HD / 2) + e);
          cs[u][h] = *(const f32x4 *)(table + 2 * h);
        }
      }
    }
  }
  if constexpr (PREP) {
    if (norms && has_items) {  // row r: head r of the group; row g: the new key
      const int r = lane & 31;
      sum.request(r == g ? krow : qrow + (r < g ? r : 0) * HD, lane);
    }
    if (vi >= 0) fresh = *(const f32x4 *)(raw.v + s * raw.v_stride + (long long)kvh * HD + 4 * vi);
  }

  // the wavefront's tiles, in the order of the kernel above
  const int last_row = PREP ? max(L - 2, 0) : L - 1;  // (in memory)
  const int rot = rotate && n > 1 ? (int)((((unsigned)(s * sh.KV + kvh)) * 2654435761u >> 12) % min((unsigned)n, rotate)) : 0;
  int kb[T];
  f32x4 vf[T][4][C::NVU];
#pragma unroll
  for (int u = 0; u < T; ++u) {
    const int k = min(wave + NW * u, n - 1) + rot;
    kb[u] = 16 * (k < n ? k : k - n);
#pragma unroll
    for (int i = 0; i < C::NKI; ++i) {  // (as issue_k_tile)
      const int slot = i * 64 + lane, row = slot / C::PPR, piece = slot % C::PPR ^ row;
      const unsigned off = (unsigned)(min(kb[u] + row, last_row) * C::ROW_BYTES + 16 * piece);
      copy_to_lds<true>(&k_lds[wave][u][i * 1024], kbase, off);
    }
  }
#pragma unroll
  for (int u = 0; u < T; ++u)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const unsigned off = (unsigned)(min(kb[u] + 4 * j + r, last_row) * C::ROW_BYTES + 16 * col);
#pragma unroll
      for (int w2 = 0; w2 < C::NVU; ++w2)
        vf[u][r][w2] = __builtin_nontemporal_load((const __attribute__((address_space(1))) f32x4 *)((uintptr_t)vbase + off + 256 * w2));
    }
  f32x4 near_bias[T];
  if constexpr (BIAS) {
    struct __attribute__((packed, aligned(4))) Four { f32x4 v; };
    const float *bias_row = db.tab + (long long)(kvh * g + cq) * db.stride + (db.origin - (L - 1));
#pragma unroll
    for (int u = 0; u < T; ++u) {
      near_bias[u] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (L - 1 - (kb[u] + 15) < db.reach) near_bias[u] = ((const Four *)(bias_row + kb[u] + 4 * j))->v;
    }
  }

  if (has_items) {
    const float inv = norms ? sum.factor(raw.eps, lane) : 1.f;
#pragma unroll
    for (int u = 0; u < kRounds; ++u) {
      const int at = threadIdx.x + 256 * u, row = at / kPieces, e = 4 * (at % kPieces);
      const float inv_row = norms ? __shfl(inv, 32 + (row < 17 ? row : 0)) : 1.f;
      if (at >= items) continue;
      if constexpr (PREP) {
        norm_rotate_quad(x[u][0], x[u][1], (row == g ? raw.k_norm : raw.q_norm) != nullptr, w[u][0], w[u][1], inv_row, cs[u][0], cs[u][1]);
        float *to = row == g ? const_cast<float *>(kbase) + (long long)(L - 1) * HD : raw.q_rot + ((long long)s * sh.H + kvh * g + row) * HD;
        *(f32x4 *)(to + e) = x[u][0];
        *(f32x4 *)(to + HD / 2 + e) = x[u][1];
        *(f32x4 *)&sm_q[row * kRow + HD / 2 + e] = x[u][1];
      }
      *(f32x4 *)&sm_q[row * kRow + e] = x[u][0];
    }
  }
  if (PREP && vi >= 0) {
    *(f32x4 *)(const_cast<float *>(vbase) + (long long)(L - 1) * HD + 4 * vi) = fresh;
    *(f32x4 *)&sm_v[4 * vi] = fresh;
  }
  __syncthreads();
  float qr[HD / 4];
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const f32x4 v = *(const f32x4 *)&sm_q[cq * kRow + 16 * i + 4 * j];
#pragma unroll
    for (int e = 0; e < 4; ++e) qr[4 * i + e] = v[e];
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // the tiles are there
  asm volatile("" ::: "memory");

  float m = -INFINITY, l = 0.f;
  f32x4 o[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < T; ++u) {
    if (wave + NW * u >= n) continue;
    const bool last = PREP && kb[u] + 16 >= L;  // the pair's last tile: nobody's key L - 1 and no value from there on is in memory
    const char *tile = k_lds[wave][u] + col * C::ROW_BYTES, *fresh_key = (const char *)&sm_q[g * kRow];
    const bool mine = last && kb[u] + col == L - 1;
    f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const f32x4 kk = *(const f32x4 *)(mine ? fresh_key + 64 * i + 16 * j : tile + (((4 * i + j) ^ col) << 4));
      s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kk.x, qr[4 * i + 0], s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kk.y, qr[4 * i + 1], s1, 0, 0, 0);
      s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kk.z, qr[4 * i + 2], s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kk.w, qr[4 * i + 3], s1, 0, 0, 0);
    }
    if (last) {
#pragma unroll
      for (int w2 = 0; w2 < C::NVU; ++w2) {
        const f32x4 v = *(const f32x4 *)&sm_v[64 * w2 + 4 * col];
#pragma unroll
        for (int r = 0; r < 4; ++r) vf[u][r][w2] = kb[u] + 4 * j + r >= L - 1 ? v : vf[u][r][w2];
      }
    }
    float sv[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
      sv[r] = (kb[u] + 4 * j + r < L) ? (BIAS ? (s0[r] + s1[r]) * c + near_bias[u][r] : s0[r] + s1[r]) : -INFINITY;
    const float mnew = fmaxf(m, max_across_quarters(fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3]))));
    const float mref = mnew == -INFINITY ? 0.f : mnew;  // (a tile of nothing but -inf)
    const float alpha = fast_exp2((m - mref) * ce);
    float p[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) p[r] = fast_exp2((sv[r] - mref) * ce);
    l = l * alpha + ((p[0] + p[1]) + (p[2] + p[3]));
    m = mnew;
#pragma unroll
    for (int i = 0; i < NT; ++i) o[i] *= alpha;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int w2 = 0; w2 < C::NVU; ++w2) {
        o[4 * w2 + 0] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[u][r][w2].x, p[r], o[4 * w2 + 0], 0, 0, 0);
        o[4 * w2 + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[u][r][w2].y, p[r], o[4 * w2 + 1], 0, 0, 0);
        o[4 * w2 + 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[u][r][w2].z, p[r], o[4 * w2 + 2], 0, 0, 0);
        o[4 * w2 + 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[u][r][w2].w, p[r], o[4 * w2 + 3], 0, 0, 0);
      }
  }

  // the wavefronts' shares meet in LDS, in their order
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);
  if (col < g) {
#pragma unroll
    for (int w2 = 0; w2 < C::NVU; ++w2)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        *(f32x4 *)&sm_o[wave][col * HD + 64 * w2 + 4 * (4 * j + r)] = f32x4{o[4 * w2][r], o[4 * w2 + 1][r], o[4 * w2 + 2][r], o[4 * w2 + 3][r]};
    if (j == 0) {
      sm_m[wave][col] = m;
      sm_l[wave][col] = l;
    }
  }
  __syncthreads();
  float *const to = out + ((long long)s * sh.H + kvh * g) * HD;
  for (int idx = threadIdx.x; idx < g * (HD / 4); idx += 64 * NW) {
    const int cc = idx / (HD / 4);
    float mm = sm_m[0][cc];
#pragma unroll
    for (int w2 = 1; w2 < NW; ++w2) mm = fmaxf(mm, sm_m[w2][cc]);
    const float mref = mm == -INFINITY ? 0.f : mm;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    float ls = 0.f;
#pragma unroll
    for (int w2 = 0; w2 < NW; ++w2) {
      const float f = fast_exp2((sm_m[w2][cc] - mref) * ce);  // 0 for a wavefront without a tile
      acc += f * *(const f32x4 *)&sm_o[w2][4 * idx];
      ls += f * sm_l[w2][cc];
    }
    *(f32x4 *)(to + 4 * idx) = f32x4{acc.x / ls, acc.y / ls, acc.z / ls, acc.w / ls};
  }
}

constexpr float kLog2e = 1.4426950408889634f;
constexpr int kDecodeWaves = 4;  // wavefronts per workgroup (eight measured 4 % slower)

// Share of each of eight consecutive spans, in thousandths of an equal share, by the XCD the
// workgroup lands on (index mod 8).  With equal spans the workgroups on odd XCDs finished
// streaming about 5 % after those on even XCDs on every box traced (3 and 5 last, 0 and 6
// first; the finer pattern differs from box to box).  SHAINET_HIP_DECODE_SHARES: eight
// numbers, or "0" for equal spans.  Not worth it for short spans.
struct Shares {
  int v[8] = {1050, 950, 1050, 950, 1050, 950, 1050, 950};
  Shares() {
    const char *env = getenv("SHAINET_HIP_DECODE_SHARES");
    if (!env) return;
    int w[8], n = 0;
    for (const char *c = env; *c && n < 8;) {
      char *end;
      const long x = strtol(c, &end, 10);
      if (end == c) break;
      w[n++] = (int)x;
      c = *end ? end + 1 : end;
    }
    for (int i = 0; i < 8; ++i) v[i] = n == 8 && w[i] >= 500 && w[i] <= 1500 ? w[i] : 1000;
  }
};
const Shares &span_shares() {
  static const Shares shares;
  return shares;
}

// Where the spans of eight consecutive workgroups begin within their 8 q tiles, from their shares.
__host__ __device__ inline void spans_from_shares(const int (&share)[8], int q, SpanTable &spans) {
  long long sum = 0, acc = 0;
  for (int i = 0; i < 8; ++i) sum += share[i];
  for (int i = 0; i <= 8; ++i) {
    spans.off[i] = q >= 32 ? (int)(acc * 8 * q / sum) : i * q;
    if (i < 8) acc += share[i];
  }
}

// Tiles per span when `total` tiles go to `wgs` workgroups: at least one per wavefront.
__host__ __device__ inline int least_span(int total, int wgs) {
  const int q = (total + wgs - 1) / wgs;
  return q < kDecodeWaves ? kDecodeWaves : q;
}
// Spans that end with the pairs (DecodePlan::align): the longest worth having for that, two tiles per
// wavefront or a quarter more than the least; shorter than the spans of unequal shares.  And whether pairs of n_s tiles
// may be cut into spans of q: a pair's last span waits for its others and merges, and with 2, 4 or 8 as a common
// divisor of the pairs' counts and 8 these meet on four, two or one of the eight XCDs.  Up to four of them on an XCD
// cost nothing, eight 0.5 to 0.9 us, which spans of one tile per wavefront are worth, 16 and more 1 to 6 us.
// Attention kernel, us, head_dim 64:   8 pairs of 40 tiles, 4 x 10 spans 8.8, 6 x 7 9.6, 5 x 8 10.6; of 32, 4 x 8 9.8, 5 x 7
// 9.6; of 160, 5 x 32 12.0, 6 x 27 10.8;   16 of 32, 4 x 8 11.5, 5 x 7 10.2; of 24, 4 x 6 9.3, 5 x 5 9.9, 6 x 4 10.7; of
// 96, 6 x 16 12.6, 7 x 14 10.6;   32 of 24, 4 x 6 9.9, 5 x 5 10.2; of 16, 4 x 4 11.4, 6 x 3 10.0; of 40, 5 x 8 16.0, 6 x 7 10.4;
// 64 of 16, 4 x 4 15.2, 6 x 3 10.9.  A pair that is one span waits for nobody.
__host__ __device__ inline int widest_aligned_span(int q) {
  const int most = q + q / 4 > 2 * kDecodeWaves ? q + q / 4 : 2 * kDecodeWaves;
  return most < 31 ? most : 31;
}
__host__ __device__ inline bool spans_may_end_with(int n_s, int q, int pairs) {
  const int count = (n_s + q - 1) / q, shared = count & 7 ? count & -count : 8;  // the common divisor
  return n_s == 0 || shared == 1 || pairs * shared <= (q == kDecodeWaves ? 64 : 32);
}
// Whether pairs of up to `longest` tiles may be a span each: nobody waits or merges then, which a few more tiles
// per wavefront are worth.  Attention kernel, us, cut as above | whole;
// head_dim 64:  8 pairs of 9 to 12 tiles 8.7 | 8.2, of 14 and 16 8.8 | 9.1;  16 of 14 9.7 | 9.1, of 16 9.1 | 9.3, of 19 9.0 | 10.2;
// 32 of 9 to 16 9.1 to 10.0 | 8.3 to 9.3, of 19 9.3 | 10.6;  64 of 9 to 16 10.0 to 11.3 | 8.8 to 9.8, of 24 11.6 | 12.0;  128 of 12
// 15.5 | 8.9, of 16 15.6 | 9.9, of 24 16.7 | 12.2, of 32 18.8 | 20.6;   head_dim 128:  8 to 64 of 9 to 16 level to a quarter
// slower;  128 of 12 17.7 | 13.0, of 16 18.7 | 15.3, of 19 and 24 level;   head_dim 96 and 256, 128 of 10 to 16 17.8 to 18.7 | 11.0 to 13.0 and
// 23.2 to 27.0 | 19.5 to 25.4.
// (Three plans stay cut although whole is level or better, because tests that state the layout name them: 8 pairs of 12 tiles 8.7 | 8.2,
// 32 of 16 10.0 | 9.3, 128 of 9 12.9 | 8.7.)
__host__ __device__ inline bool whole_pairs(int longest, int q, int hd, int pairs) {
  if (longest <= q) return false;
  if (longest <= widest_aligned_span(q)) return true;
  if (pairs >= 128) return longest >= 10 && longest <= (hd <= 64 ? 24 : 16);
  return hd <= 64 && longest <= (pairs >= 16 ? 15 : 11);
}
// And whether that is tried in front of the cuts that end with the pairs: not where a few long pairs would be what the launch takes.
// 16 sequences of 8 kv heads, some of them longer, us, such a cut | whole;  four rows x heads of 64:  1 of 16 tiles and 15 of 1 9.9 | 9.3,
// 1 of 20 and 15 of 8 level, of 24 and 1 10.2 | 11.1 (heads of 16 to 48: 9.2 | 10.4), 4 of 24 and 12 of 8 10.7 | 11.3, 8 of 24 and 8 of 1
// level;  heads of 96:  1 of 10 and 15 of 1 9.7 | 10.6, 1 of 16 11.2 | 12.3;  of 128:  11.1 | 11.8, 12.4 | 13.2 (but 8 of 10 and 8 of 4, which
// take all 256 workgroups, 12.6 | 12.2);  of 256:  12.1 | 16.5, 15.2 | 20.7.  More rows make the merge dearer:  8 x 64 of 24 and 1 10.6 |
// 10.5, 16 x 64 13.5 | 11.1;  8 x 128 of 16 and 1 12.2 | 12.2 and 14.4 | 14.2, 16 x 128 16.1 | 14.1;  8 x 256 18.6 | 23.4, 16 x 256 24.1 | 27.3.
// Where no cut ends with the pairs, whole is the better way in any case:  1 of 16 and 15 of 8 15.3 | 9.5, 18.6 | 12.5, 17.8 | 13.7, 24 | 23.7.
__host__ __device__ inline bool whole_first(int longest, int q, int hd, int cols) {
  return longest <= widest_aligned_span(q) || (hd <= 64 && longest <= 16) || (hd <= 128 && cols >= 8);
}

// Tiles per wavefront of decode_rows_kernel, or 0: not a call for it.  (Longer pairs would take more rounds of a wavefront's tiles, 1 us each, which the
// kernel above overlaps with their loads; heads of 128 take twice the registers.)
int row_tiles(const SeqTable &st, const Shape &sh, const DecodePlan &p, const DistanceBias *bias) {
  if ((sh.hd != 64 && sh.hd != 128) || p.align <= 1 || (bias && bias->v_hd != sh.hd)) return 0;
  int most = 0;
  for (int s = 0; s < st.n_seqs; ++s) {
    const int n = (st.start_pos[s] + 16) / 16;
    if (st.n_new[s] != 1 || st.tok_off[s] != s || n > p.align || (s && st.slot[s] == st.slot[s - 1])) return 0;
    most = n > most ? n : most;
  }
  const int tiles = (most + kDecodeWaves - 1) / kDecodeWaves;
  return tiles <= (sh.hd == 64 ? kRowTiles<64> : kRowTiles<128>) ? tiles : 0;
}

struct ShareArg {
  int v[8];
};

// plan_decode on the device for one new row per sequence: one wavefront, lane s looks after
// sequence s.  Reads the cached lengths, writes the record the step's prep and decode kernels
// read, and adds the step's rows to the lengths.
__global__ __launch_bounds__(64) void decode_plan_kernel(int *__restrict__ lens, int n_seqs, Shape sh, int rope_positions,
                                                         ShareArg shares, DecodeDevicePlan *__restrict__ out,
                                                         int *error) {
  const int s = threadIdx.x;
  const bool mine = s < n_seqs;
  const int start = mine ? lens[s] : 0;
  const bool fits = !mine || (start >= 0 && start + 1 <= sh.cap && start + 1 <= rope_positions);
  if (!__all(fits)) {  // nothing is appended: the lengths stay as they are
    if (s == 0) {
      out->st.n_seqs = n_seqs;
      out->tiles_per_wg = 0;
      out->total_tiles = 0;
      out->align = 1;
      out->align_by = 0;
      out->skip = 1;
      spans_from_shares(shares.v, 0, out->spans);  // all zero: no workgroup finds tiles
      if (*error == 0) *error = 2;  // a pending 1 (a given-up wait) is the graver report and stays
    }
    return;
  }
  const int n_s = mine ? (start + 1 + 15) >> 4 : 0;
  auto prefix = [&](int x) {  // inclusive prefix sum over the lanes
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int up = __shfl_up(x, o);
      if (s >= o) x += up;
    }
    return x;
  };
  int tiles = sh.KV * n_s;
  int incl = prefix(tiles), total = __shfl(incl, 63), q = least_span(total, kDevicePlanWorkgroups), align = 1;
  int longest = n_s;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) longest = max(longest, __shfl_xor(longest, o));
  const int widest = widest_aligned_span(q);
  auto takes = [&](int a) {
    if (!__all(spans_may_end_with(n_s, a, n_seqs * sh.KV)) ||
        __shfl(prefix(sh.KV * ((n_s + a - 1) / a)), 63) > kDevicePlanWorkgroups)
      return false;
    q = align = a;
    tiles = sh.KV * padded_tiles(n_s, a);
    incl = prefix(tiles);
    total = __shfl(incl, 63);
    return true;
  };
  const bool whole = whole_pairs(longest, q, sh.hd, n_seqs * sh.KV), first = whole && whole_first(longest, q, sh.hd, sh.g);
  bool laid = first && takes(longest);
  for (int a = q; a <= widest && !laid; ++a) laid = takes(a);
  if (whole && !first && !laid) takes(longest);
  if (mine) {
    out->st.slot[s] = s;
    out->st.start_pos[s] = start;
    out->st.n_new[s] = 1;
    out->st.tok_off[s] = s;
    out->st.work_off[s] = incl - tiles;
    lens[s] = start + 1;
  }
  if (s == 0) {
    out->st.n_seqs = n_seqs;
    out->st.tok_off[n_seqs] = n_seqs;
    out->st.work_off[n_seqs] = total;
    out->tiles_per_wg = q;
    out->align = align;
    out->align_by = align_factor(align);
    out->total_tiles = total;
    out->skip = 0;
    spans_from_shares(shares.v, q, out->spans);
  }
}

}  // namespace

DecodePlan plan_decode(SeqTable &st, const Shape &sh, int wg_target, bool aligned) {
  DecodePlan p;
  auto lay_out = [&](int align) {
    p.align = align;
    st.work_off[0] = 0;
    for (int s = 0; s < st.n_seqs; ++s)
      st.work_off[s + 1] = st.work_off[s] + sh.KV * padded_tiles((st.start_pos[s] + st.n_new[s] + 15) / 16, align);
    p.total_tiles = st.work_off[st.n_seqs];
  };
  lay_out(1);
  // One workgroup on each of the 256 compute units.  Its four wavefronts keep 64 KiB
  // of K and V in flight, 16 MiB over the chip, which saturates HBM; twice as many
  // workgroups only double the partials to merge and the arrivals at each pair's
  // counter (measured: 4 to 10 % slower from batch 1 x 4096 to batch 4 x 32768).
  if (wg_target < 1) wg_target = 256;
  int q = least_span(p.total_tiles, wg_target);
  // Spans that end with the pairs, where that takes no more workgroups: a span that runs from one pair
  // into the next is two segments behind each other with a merge in between.  The attention kernel, 8 kv heads of 64
  // (128), us, laid end to end : this way: one sequence of 100 keys 10.7 : 7.3 (12.3 : 9.1), whole pairs; of 512 10.1 : 10.2
  // (11.1 : 11.0), of 528 10.7 : 9.8 (12.7 : 10.8), of 640 9.2 : 9.7 (10.4 : 10.6), of 1040 10.6 : 9.7 (13.7 : 12.4); four
  // of 640 16.2 : 10.9 (18.1 : 12.6); 16 of 100 13.7 : 7.2 (16.0 : 10.7).
  int longest = 0;
  p.cols = 0;
  for (int s = 0; s < st.n_seqs; ++s) {
    const int n_s = (st.start_pos[s] + st.n_new[s] + 15) / 16;
    longest = n_s > longest ? n_s : longest;
    p.cols = st.n_new[s] * sh.g > p.cols ? st.n_new[s] * sh.g : p.cols;
  }
  const int widest = widest_aligned_span(q);
  auto takes = [&](int a) {
    long long wgs = 0;
    bool fits = true;
    for (int s = 0; s < st.n_seqs; ++s) {
      const int n_s = (st.start_pos[s] + st.n_new[s] + 15) / 16;
      fits = fits && spans_may_end_with(n_s, a, st.n_seqs * sh.KV);
      wgs += (long long)sh.KV * ((n_s + a - 1) / a);
    }
    if (!fits || wgs > wg_target) return false;
    q = a;
    lay_out(a);
    return true;
  };
  const bool whole = aligned && whole_pairs(longest, q, sh.hd, st.n_seqs * sh.KV), first = whole && whole_first(longest, q, sh.hd, p.cols);
  bool laid = first && takes(longest);
  for (int a = q; aligned && a <= widest && !laid; ++a) laid = takes(a);
  if (whole && !first && !laid) takes(longest);
  p.tiles_per_wg = q;
  spans_from_shares(span_shares().v, q, p.spans);
  // the first workgroup count whose spans cover the stream
  p.n_wgs = (p.total_tiles + q - 1) / q;
  auto begin_of = [&](int w) { return (w >> 3) * 8 * q + p.spans.off[w & 7]; };
  while (p.n_wgs > 1 && begin_of(p.n_wgs - 1) >= p.total_tiles) --p.n_wgs;
  while (begin_of(p.n_wgs) < p.total_tiles) ++p.n_wgs;
  p.n_slots = p.n_wgs + st.n_seqs * sh.KV;
  return p;
}

size_t decode_flag_words(const DecodePlan &p) { return (size_t)p.n_slots * kDecodeWaves; }

// The head dimension the split-K kernel's tiles are laid out for: 64, 128 or 256 (0: none fits).
int decode_tile_head_dim(int hd) {
  if (hd < 4 || (hd & 3) || hd > 256) return 0;
  return hd <= 64 ? 64 : hd <= 128 ? 128 : 256;
}

size_t decode_partial_floats(const Shape &sh, const DecodePlan &p, int v_hd) {
  return (size_t)p.n_slots * p.cols * (decode_tile_head_dim(v_hd > sh.hd ? v_hd : sh.hd) + 2);
}

hipError_t launch_decode_plan(int *lens, int n_seqs, const Shape &sh, int rope_positions, DecodeDevicePlan *out,
                              int *error, hipStream_t stream) {
  if (!lens || !out || !error || n_seqs < 1 || n_seqs > kMaxSeqs) return hipErrorInvalidValue;
  ShareArg shares;
  for (int i = 0; i < 8; ++i) shares.v[i] = span_shares().v[i];
  hipLaunchKernelGGL(decode_plan_kernel, dim3(1), dim3(64), 0, stream, lens, n_seqs, sh, rope_positions, shares, out,
                     error);
  return hipGetLastError();
}

bool decode_prepares(const PrepArgs &a, const SeqTable &st, const Shape &sh, const DecodePlan &p, const float *out) {
  static const bool off = getenv("SHAINET_HIP_NO_FUSED_PREP") != nullptr;
  if (off || (sh.hd != 64 && sh.hd != 128) || p.align <= 1 || a.b_q || a.b_k || a.b_v || !a.rope_tab || !a.q_rot) return false;
  for (int s = 0; s < st.n_seqs; ++s)  // (two entries of one sequence: the second one's keys include the first one's row)
    if (st.n_new[s] != 1 || (s && st.slot[s] == st.slot[s - 1])) return false;
  if (((uintptr_t)a.q | (uintptr_t)a.k | (uintptr_t)a.v | (uintptr_t)a.q_norm | (uintptr_t)a.k_norm | (uintptr_t)a.rope_tab |
       (uintptr_t)a.q_rot | (uintptr_t)a.kc | (uintptr_t)a.vc) & 15 || (a.q_stride | a.k_stride | a.v_stride) & 3)
    return false;
  auto apart = [&](const float *x, long long stride, int width) {  // x's rows and out's
    const float *x_end = x + (st.n_seqs - 1) * stride + width, *out_end = out + (long long)st.n_seqs * sh.H * sh.hd;
    return (uintptr_t)x_end <= (uintptr_t)out || (uintptr_t)out_end <= (uintptr_t)x;
  };
  return apart(a.q, a.q_stride, sh.H * sh.hd) && apart(a.k, a.k_stride, sh.KV * sh.hd) && apart(a.v, a.v_stride, sh.KV * sh.hd);
}

hipError_t launch_decode(const DecodeArgs &d, const SeqTable &st, const Shape &sh, const DecodePlan &p, float scale,
                         hipStream_t stream, hipEvent_t before, hipEvent_t after, const DecodeDevicePlan *dev,
                         const DistanceBias *bias, const PrepArgs *prep) {
  const DistanceBias db = bias ? *bias : DistanceBias{};
  const PrepArgs raw = prep ? *prep : PrepArgs{};
  if (prep && (dev || bias || !decode_prepares(*prep, st, sh, p, d.out))) return hipErrorInvalidValue;
  if (st.n_seqs < 1 || st.n_seqs > kMaxSeqs || sh.g < 1 || sh.g > 16 || sh.H != sh.KV * sh.g ||
      !decode_tile_head_dim(sh.hd) || p.n_wgs < 1 || !d.partials || !d.part_flag || !d.error)
    return hipErrorInvalidValue;
  if (dev) {
    if (p.n_wgs != kDevicePlanWorkgroups || p.n_slots != device_plan_slots(st.n_seqs, sh.KV) || p.cols < sh.g)
      return hipErrorInvalidValue;
  } else {
    if (p.tiles_per_wg < 1) return hipErrorInvalidValue;
    for (int s = 0; s < st.n_seqs; ++s)
      if (st.n_new[s] < 1 || st.n_new[s] * sh.g > 16 || st.n_new[s] * sh.g > p.cols || st.start_pos[s] < 0 ||
          st.start_pos[s] + st.n_new[s] > sh.cap || st.slot[s] < 0)
        return hipErrorInvalidValue;
  }
  if (!d.q_rot) return hipErrorInvalidValue;
  if (bias && (dev || !db.tab || db.v_hd < 4 || (db.v_hd & 3) || (db.q_stride & 3) || db.v_hd > 256)) return hipErrorInvalidValue;
  unsigned *flag_set = d.flag_set ? d.flag_set : d.part_flag;
  const int spin_limit = d.spin_limit > 0 ? d.spin_limit : kFlagSpinLimit;
  float *part_o = d.partials;
  const int tile_hd = decode_tile_head_dim(bias && db.v_hd > sh.hd ? db.v_hd : sh.hd);
  float *part_ml = d.partials + (size_t)p.n_slots * p.cols * tile_hd;
  const float c = scale * kLog2e;
  // before / after (nullable) receive the kernel's own first and last clock reading, not the
  // time at which the stream reached them: what is between two kernels stays out
  dim3 grid((unsigned)p.n_wgs), block(64 * kDecodeWaves);
  ReadAhead ah = {nullptr, 0, 0, 0};
  if (d.ahead.w && d.ahead.wgs > 0 && !dev && !bias && !before && !after && (sh.hd == 64 || sh.hd == 128) && d.ahead.k >= 256 &&
      (d.ahead.k & 255) == 0 && d.ahead.n > 0) {
    ah.w = d.ahead.w;
    ah.k = d.ahead.k;
    ah.n = d.ahead.n;
    ah.first_wg = (p.n_wgs + 7) / 8 * 8;
    const int most = (d.ahead.n + 3) / 4;
    grid.x = (unsigned)(ah.first_wg + (d.ahead.wgs < most ? d.ahead.wgs : most));
  }
  // SHAINET_HIP_DECODE_NO_ROTATE: every workgroup walks its segments from their first tile (for
  // comparison); SHAINET_HIP_DECODE_ROTATE=n: starts spread over the first n tiles only
  static const unsigned rotate = getenv("SHAINET_HIP_DECODE_NO_ROTATE") ? 0u
                                 : getenv("SHAINET_HIP_DECODE_ROTATE")
                                     ? (unsigned)atoi(getenv("SHAINET_HIP_DECODE_ROTATE"))
                                     : 0x7fffffffu;
  if (const int tiles = dev ? 0 : row_tiles(st, sh, p, bias)) {
    RowSeqs seqs = {};
    for (int s = 0; s < st.n_seqs; ++s) {
      seqs.start[s] = st.start_pos[s];
      seqs.slot[s] = st.slot[s];
    }
    if (st.n_seqs > 1) ah.w = nullptr;
    grid = dim3(ah.w ? grid.x : (unsigned)sh.KV, (unsigned)st.n_seqs);
#define SHAINET_ROWS_LAUNCH(HD_, T_, MODE_)                                                                                          \
  SHAINET_LAUNCH_TIMED((decode_rows_kernel<HD_, T_, MODE_>), grid, block, 0, stream, before, after, d.q_rot, d.kc, d.vc, d.out, seqs, \
                       sh, c, rotate, ah, db, raw)
#define SHAINET_ROWS_LAUNCH_T(HD_, T_)           \
  do {                                           \
    if (prep)                                    \
      SHAINET_ROWS_LAUNCH(HD_, T_, kRowsPrep);   \
    else if (bias)                               \
      SHAINET_ROWS_LAUNCH(HD_, T_, kRowsBias);   \
    else                                         \
      SHAINET_ROWS_LAUNCH(HD_, T_, kRowsPlain);  \
  } while (0)
    if (sh.hd == 64 && tiles == 1)
      SHAINET_ROWS_LAUNCH_T(64, 1);
    else if (sh.hd == 64 && tiles == 2)
      SHAINET_ROWS_LAUNCH_T(64, 2);
    else if (sh.hd == 64)
      SHAINET_ROWS_LAUNCH_T(64, 3);
    else if (tiles == 1)
      SHAINET_ROWS_LAUNCH_T(128, 1);
    else
      SHAINET_ROWS_LAUNCH_T(128, 2);
#undef SHAINET_ROWS_LAUNCH_T
#undef SHAINET_ROWS_LAUNCH
    return hipGetLastError();
  }
#define SHAINET_DECODE_LAUNCH(HD_, DEV_, PAD_)                                                                      \
  SHAINET_LAUNCH_TIMED((decode_splitk_kernel<HD_, kDecodeWaves, DEV_, PAD_>), grid, block, 0, stream, before,      \
                       after, d.q_rot, d.kc, d.vc, d.out, part_o, part_ml, d.part_flag, flag_set, spin_limit,       \
                       d.error, st, sh, p.tiles_per_wg, p.spans, p.total_tiles, p.align, align_factor(p.align), p.n_slots, p.cols, c, rotate, dev, ah, db, raw)
#define SHAINET_DECODE_LAUNCH_HD(HD_, PAD_) \
  do {                                      \
    if (dev)                                \
      SHAINET_DECODE_LAUNCH(HD_, true, PAD_);  \
    else                                    \
      SHAINET_DECODE_LAUNCH(HD_, false, PAD_); \
  } while (0)
#define SHAINET_DECODE_LAUNCH_BIAS(HD_)                                                                             \
  SHAINET_LAUNCH_TIMED((decode_splitk_kernel<HD_, kDecodeWaves, false, true, false, true>), grid, block, 0, stream, \
                       before, after, d.q_rot, d.kc, d.vc, d.out, part_o, part_ml, d.part_flag, flag_set,           \
                       spin_limit, d.error, st, sh, p.tiles_per_wg, p.spans, p.total_tiles, p.align, align_factor(p.align), p.n_slots, p.cols, c,   \
                       rotate, dev, ah, db, raw)
#define SHAINET_DECODE_LAUNCH_PREP(HD_, AHEAD_)                                                                      \
  SHAINET_LAUNCH_TIMED((decode_splitk_kernel<HD_, kDecodeWaves, false, false, AHEAD_, false, true>), grid, block, 0,  \
                       stream, before, after, d.q_rot, d.kc, d.vc, d.out, part_o, part_ml, d.part_flag, flag_set,    \
                       spin_limit, d.error, st, sh, p.tiles_per_wg, p.spans, p.total_tiles, p.align,                 \
                       align_factor(p.align), p.n_slots, p.cols, c, rotate, dev, ah, db, raw)
  if (prep && sh.hd == 64 && ah.w)
    SHAINET_DECODE_LAUNCH_PREP(64, true);
  else if (prep && sh.hd == 64)
    SHAINET_DECODE_LAUNCH_PREP(64, false);
  else if (prep && ah.w)
    SHAINET_DECODE_LAUNCH_PREP(128, true);
  else if (prep)
    SHAINET_DECODE_LAUNCH_PREP(128, false);
  else if (bias && tile_hd == 64)
    SHAINET_DECODE_LAUNCH_BIAS(64);
  else if (bias && tile_hd == 128)
    SHAINET_DECODE_LAUNCH_BIAS(128);
  else if (bias)
    SHAINET_DECODE_LAUNCH_BIAS(256);
  else if (ah.w && sh.hd == 64)
    hipLaunchKernelGGL((decode_splitk_kernel<64, kDecodeWaves, false, false, true>), grid, block, 0, stream, d.q_rot, d.kc,
                       d.vc, d.out, part_o, part_ml, d.part_flag, flag_set, spin_limit, d.error, st, sh, p.tiles_per_wg,
                       p.spans, p.total_tiles, p.align, align_factor(p.align), p.n_slots, p.cols, c, rotate, dev, ah, db, raw);
  else if (ah.w)
    hipLaunchKernelGGL((decode_splitk_kernel<128, kDecodeWaves, false, false, true>), grid, block, 0, stream, d.q_rot, d.kc,
                       d.vc, d.out, part_o, part_ml, d.part_flag, flag_set, spin_limit, d.error, st, sh, p.tiles_per_wg,
                       p.spans, p.total_tiles, p.align, align_factor(p.align), p.n_slots, p.cols, c, rotate, dev, ah, db, raw);
  else if (sh.hd == 64)
    SHAINET_DECODE_LAUNCH_HD(64, false);
  else if (sh.hd == 128)
    SHAINET_DECODE_LAUNCH_HD(128, false);
  else if (tile_hd == 64)
    SHAINET_DECODE_LAUNCH_HD(64, true);
  else if (tile_hd == 128)
    SHAINET_DECODE_LAUNCH_HD(128, true);
  else
    SHAINET_DECODE_LAUNCH_HD(256, true);
#undef SHAINET_DECODE_LAUNCH_PREP
#undef SHAINET_DECODE_LAUNCH_BIAS
#undef SHAINET_DECODE_LAUNCH_HD
#undef SHAINET_DECODE_LAUNCH
  return hipGetLastError();
}

}  // namespace shainet
