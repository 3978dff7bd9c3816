// Row-major fp32 product y[T,N] = x[T,K] W[K,N] (+ res) for gfx950, for five rows and more: the
// projections of a prefill (llama_block.cr:253-255, 298; swiglu_ff.cr:76-91), where the
// reference's GPU branch calls cuBLAS SGEMM (llama_block.cr:726-768, cuda.cr:237-247) and its CPU
// branch SimpleMatrix#* (simple_matrix.cr:61-74).
//
// The product runs on the bf16 matrix cores, each operand as the exact sum of three bf16 numbers
// (split_mfma.hpp).  A workgroup of 2 x WN wavefronts owns a tile of 64 MB rows and 64 WN columns of y; each
// wavefront owns MB x 2 blocks of 32 x 32 and the workgroup walks K in steps of 16.
// A step's tiles go global memory -> registers (one or two steps ahead) -> split -> LDS (two stages, one
// barrier per step), where the fragments of an MFMA lie as it takes them: unit [part][octet of k][row or
// column] of 16 bytes, so that 32 lanes read 512 consecutive bytes.
//   x: a thread takes an octet of k of a row, or half of one;
//   W: a thread takes 8 rows of one column, so that the pairs of k that share a register come from two of
//      its registers and nothing has to be transposed.  Column c of a wavefront's 64 lies in block c % 2 at
//      place c / 2: a lane's two blocks are neighbouring columns of y (8-byte stores, 256 bytes a row).
// Tile loads take a scalar base that moves along K plus a per-thread 32-bit offset.
// W whose values are bf16 numbers (a checkpoint's, most often): the other two of its parts are zeros, and the three
// products with them add nothing.  They are left out: sgemm_wide_kernel, sgemm_stream_kernel.
// What bounds the others: large shapes the power the card may draw.  4096 rows of 2048 -> 16384 run at 232 TFLOP/s
// with N(0, 1) operands and at 295 with zeros (71 % of the six products' rate); with four wavefronts on
// 128 x 128 tiles it was 183 and 252, so the large tile, which reads LDS 3/4 as often and splits half as much
// per product, is worth more than a better schedule (an order forced between MFMAs and splits, three
// workgroups per compute unit: 1 to 6 % slower).  The fp32 instruction it replaces, in tiles of 128 x 128,
// reached 137.  Small shapes: a launch, the first loads' way, and the kernel that adds the pieces.
//
// Work is counted in units of one K step of one tile.  When the tiles do not fill whole rounds of
// the chip, the units are dealt out evenly instead: a workgroup takes
// a contiguous run of units, which may end inside a tile (it leaves that piece as a partial product
// in its own slot of a scratch array and marks the slot's flag word) and may begin inside one (it
// then finishes that tile: waits for the flag words of the workgroups that hold the tile's earlier
// pieces, adds their partial products to its own in a fixed order and stores y).  Which
// workgroup holds which piece depends on the shape only, so results do not depend on scheduling.
// A workgroup waits only for workgroups with a lower index, which were started before it and wait
// for nobody in turn while they compute the piece it needs (every workgroup computes the piece it
// leaves unfinished first).  That serves shapes where a tile is shared by two or three workgroups.
// Few tiles with a long K (512 rows of the 8192 -> 2048 down projection: 64 tiles for 256 compute
// units) are cut into more pieces per tile; one workgroup adding them one after the other would take
// longer than the product, so there every workgroup leaves its piece in its slot and a second
// kernel, with the whole chip, adds the pieces in a fixed order (and the residual).
#include "gemm_kernel.hpp"

#include "attn_kernels.hpp"
#include "lds_copy.hpp"
#include "split_mfma.hpp"

#include <math.h>
#include <stdint.h>
#include <stdlib.h>

namespace shainet {

namespace {

constexpr int TK = 16, kFewStep = 32, kWideStep = 32;  // K of a step: tiles of three-part weights, of 32 rows, large tiles of one-part weights

// A partial product is read by a workgroup that may sit on another XCD, whose L2 is not kept
// coherent with this one's for ordinary accesses: the store is written through to memory.
// (The compiler does not see a store in this text: the registers of v must not be written again
// before the store has read them, so callers keep every value they store in registers of its own
// until they have waited for the stores.)
__device__ __forceinline__ void coherent_store4(float *p, f32x4 v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" : : "v"(p), "v"(v) : "memory");
}

struct GemmArgs {
  const float *x;
  long long xs;
  const unsigned short *planes;  // instead of x: its parts, lifted, [3][K / 32][T][32] (split_mfma.hpp)
  const float *w;
  float *y;
  const float *res;  // nullable: y = res + x W
  const float *bias;  // nullable: y = act(x W + bias)
  Activation act;
  float *partials;   // [workgroups][a tile]: the piece a workgroup leaves unfinished
  unsigned *flags;   // [workgroups], zero between launches
  unsigned *flag_set;  // where a piece is marked complete: `flags`, or elsewhere in the test of the give-up path
  int spin_limit;    // polls before a wait for a flag word is given up
  int *error;        // set to 1 then
  int T, K, N, tiles_m;
  int steps;            // K steps of 16 per tile
  int group_bits;       // workgroup id -> group id & (groups - 1), place id >> group_bits
  int tiles_per_group;  // a group's workgroups share a contiguous run of tiles (row tiles fastest)
  int quota;            // units per workgroup
  int pieces;           // 0: a workgroup's run of units starts where the one before it ends; > 0: every tile
                        // is cut into this many pieces of `quota` steps, a workgroup each, all left in their slots
};

// v: columns col and col + 1 of x W; rows past the last one are dropped
__device__ __forceinline__ void store_pair(const GemmArgs &g, int row, int col, f32x2 v) {
  if (row >= g.T) return;
  const long long o = (long long)row * g.N + col;
  if (g.bias) {
    const f32x2 b = *(const f32x2 *)(g.bias + col);
    v = f32x2{activate(g.act, v.x + b.x), activate(g.act, v.y + b.y)};
  }
  if (g.res) {
    const f32x2 r = *(const f32x2 *)(g.res + o);
    v = f32x2{r.x + v.x, r.y + v.y};
  }
  *(f32x2 *)(g.y + o) = v;
}

// Four registers of a lane's sums, number r of its 4 MB NB: with one block its column in four rows, with two blocks beside
// each other its two columns in two rows, with four its four columns in one row.  row_of: the first of these rows.
template <int NB>
__device__ __forceinline__ int row_of(int r) {
  return NB == 1 ? 32 * (r >> 2) + 8 * (r & 3) : NB == 2 ? 32 * (r >> 3) + 8 * ((r & 7) >> 1) + 2 * (r & 1) : 32 * (r >> 4) + 8 * ((r & 15) >> 2) + (r & 3);
}
template <int NB>
__device__ __forceinline__ void store_four(const GemmArgs &g, int row0, int col, int r, f32x4 v) {
  const int row = row0 + row_of<NB>(r);
  if constexpr (NB == 1) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (row + i >= g.T) return;
      const long long o = (long long)(row + i) * g.N + col;
      float y = v[i];
      if (g.bias) y = activate(g.act, y + g.bias[col]);
      g.y[o] = g.res ? g.res[o] + y : y;
    }
  } else if constexpr (NB == 2) {
    store_pair(g, row, col, f32x2{v.x, v.y});
    store_pair(g, row + 1, col, f32x2{v.z, v.w});
  } else {
    if (row >= g.T) return;
    const long long o = (long long)row * g.N + col;
    if (g.bias) {
      const f32x4 b = *(const f32x4 *)(g.bias + col);
      v = f32x4{activate(g.act, v.x + b.x), activate(g.act, v.y + b.y), activate(g.act, v.z + b.z), activate(g.act, v.w + b.w)};
    }
    if (g.res) v = *(const f32x4 *)(g.res + o) + v;
    *(f32x4 *)(g.y + o) = v;
  }
}

// The piece of a tile that a workgroup's run leaves unfinished: to its slot, which is marked complete.
template <int OUT>
__device__ __forceinline__ void leave_piece(const GemmArgs &g, float *slot, int step, const f32x4 (&out)[OUT]) {
  __builtin_amdgcn_sched_barrier(0);  // all of out[] is in place before the first store is issued
#pragma unroll
  for (int r = 0; r < OUT; ++r) coherent_store4(slot + r * step, out[r]);
  // the stores are acknowledged (s_waitcnt vmcnt(0): the barrier alone does not wait for them)
  // before the piece is marked complete
  __builtin_amdgcn_s_waitcnt(0x0F70);
  __syncthreads();
  if (threadIdx.x == 0) __hip_atomic_store(g.flag_set + blockIdx.x, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Adds the tile's earlier pieces, those of the `before` places from `first` on (lower indices, waiting for nobody), to out[].
template <int OUT>
__device__ __forceinline__ void add_earlier_pieces(const GemmArgs &g, int group, int first, int before, long long slot_floats, int in_slot,
                                                   int step, f32x4 (&out)[OUT]) {
  const int lane = threadIdx.x & 63;
  if (threadIdx.x < 64) {
    for (int spins = 0;; ++spins) {
      bool ok = true;
      for (int i = lane; i < before; i += 64)
        ok = ok && __hip_atomic_load(g.flags + (((first + i) << g.group_bits) | group), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u;
      if (__all(ok)) {
        for (int i = lane; i < before; i += 64)
          __hip_atomic_store(g.flags + (((first + i) << g.group_bits) | group), 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        break;
      }
      if (spins >= g.spin_limit) {
        if (lane == 0) *g.error = 1;
        break;
      }
      __builtin_amdgcn_s_sleep(2);
    }
  }
  __syncthreads();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  // ((own piece + piece 0) + piece 1) + ...
  const float *piece = g.partials + (long long)((first << g.group_bits) | group) * slot_floats + in_slot;
  const long long piece_step = slot_floats << g.group_bits;
  for (int i = 0; i < before; ++i) {
#pragma unroll
    for (int r0 = 0; r0 < OUT; r0 += 16) {
      f32x4 v[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) v[r] = *(const f32x4 *)(piece + i * piece_step + (r0 + r) * step);
      __builtin_amdgcn_sched_barrier(0);  // all loads in flight before the first sum waits
#pragma unroll
      for (int r = 0; r < 16; ++r) out[r0 + r] += v[r];
    }
  }
}

// WM x WN wavefronts of MB x 2 blocks.  Units of 16 bytes in a stage of LDS.  A part of x: two octets of TM rows, four
// units apart from a multiple of 16 (a wavefront writes both octets of 32 rows); a part of W: two octets of WN
// wavefronts' two blocks of 32 columns, four units of padding behind each (neighbouring columns lie in both).
template <int WM, int WN, int MB>
struct Stage {
  static constexpr int kOctX = 32 * WM * MB + 4, kPartX = 2 * kOctX;
  static constexpr int kOctW = 72 * WN, kPartW = 2 * kOctW;
  static constexpr int kUnits = 3 * (kPartX + kPartW);
};

// SWIGLU: W is gate | up, y is [T, N / 2], silu(gate) * up.  A lane then holds both halves of its column of y: hidden column h of the tile's TN / 2.
__device__ __forceinline__ void store_swiglu(const GemmArgs &g, int row0, int h, int r, f32x4 v) {
  const int row = row0 + row_of<2>(r), N = g.N / 2;
  if (row >= g.T) return;
  float *const y = g.y + (long long)row * N + h;
  y[0] = swiglu(v.x, v.y);
  const float second = swiglu(v.z, v.w);
  if (row + 1 < g.T) y[N] = second;
}

// W of three parts.  GUARD: K need not be a multiple of 16 (pieces beyond its end are zeros).
// SWIGLU (no pieces): the activation, a launch of 10.6 us behind 512 rows of 2048 -> 2 x 8192 and of 32.5 behind 2048 rows, between which the
// wide rows were written and read again, happens where the sums are.  Us, both launches | this: 512 rows 113.8 | 99.4, 2048 rows
// 408 | 358, 777 rows of 1024 -> 2 x 1024 in tiles of sgemm_stream_kernel 29.5 | 22.8; weights of three parts: a block of width 2048 401 | 392 at 384
// rows, 461 | 451 at 512, of width 1024 264 | 255 at 777; none in tiles of 256 x 256 (gemm_takes_next).
template <int WM, int WN, int MB, bool GUARD, bool SWIGLU>
__global__ __launch_bounds__(64 * WM * WN, 2) void sgemm_split_kernel(const GemmArgs g) {
  constexpr int NB = 2, TM = 32 * WM * MB, TN = 32 * WN * NB, NT = 64 * WM * WN;
  constexpr int NX = 4 * TM / NT;  // float4 of the x tile per thread
  constexpr int kSets = TM == 256 ? 1 : 2;
  using S = Stage<WM, WN, MB>;
  static_assert(2 * TN == NT, "a thread stages an octet of W");
  static_assert(NX == 2 || NX == 1, "a thread stages an octet of x, or half of one");
  __shared__ __attribute__((aligned(16))) u32x4 lds[2][S::kUnits];

  // Workgroups go to the eight XCDs round-robin by index: the workgroups of a group (index modulo
  // the group count, a power of two up to 8) stay on the same XCDs and share a run of tiles, whose
  // operands and partial products they find in those XCDs' L2.
  const int group = blockIdx.x & ((1 << g.group_bits) - 1), place = blockIdx.x >> g.group_bits;
  const int steps = g.steps;
  int u0 = place * g.quota, u1 = min(u0 + g.quota, g.tiles_per_group * steps);
  if (g.pieces) {
    const int t = place / g.pieces;
    u0 = t * steps + (place - t * g.pieces) * g.quota;
    u1 = t < g.tiles_per_group ? min(u0 + g.quota, (t + 1) * steps) : u0;
  }
  if (u0 >= u1) return;
  const int t_first = u0 / steps, t_last = (u1 - 1) / steps;
  const bool leaves_piece = u1 < (t_last + 1) * steps;  // the run ends inside tile t_last

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int T = g.T, K = g.K, N = g.N;
  const long long w_step = (long long)TK * N * 4;

  for (int visit = 0; visit <= t_last - t_first; ++visit) {
    // the tile this run leaves unfinished comes first: the workgroup that finishes it needs the piece
    const int t = leaves_piece ? (visit == 0 ? t_last : t_first + visit - 1) : t_first + visit;
    const int s_begin = t == t_first ? u0 - t_first * steps : 0;
    const int s_end = t == t_last ? u1 - t_last * steps : steps;
    const int tile = group * g.tiles_per_group + t;
    const int tm = tile % g.tiles_m, tn = tile / g.tiles_m;
    const int m0 = tm * TM, n0 = tn * TN;
    const int k_begin = s_begin * TK, k_end = min(K, s_end * TK);
    const int nk = s_end - s_begin;

    // (what follows from the thread's number is worked out per tile, or the compiler keeps it in scratch memory over the
    // tile's end and the loads of the first step wait for it.  128 x 128 has the registers, and without them puts all of a step's
    // splits in front of its MFMAs: 200 rows of 8192 -> 1024, a workgroup a compute unit, 30 -> 35 us)
    int tid = threadIdx.x;
    if constexpr (WN == 4) asm volatile("" : "+v"(tid));
    const int lane = tid & 63;
    const int ln = lane & 31, j = lane >> 5;

    // staging: x: octet tid % 2 of row tid / 2, or half of one, quarter tid % 4 of row tid / 4; W: octet tid / TN
    // of column tid % TN
    const int xrow = NX == 1 ? tid >> 2 : tid >> 1;
    const int xk = NX == 1 ? 4 * (tid & 3) : 8 * (tid & 1);
    int wcol = tid & (TN - 1), w_from = min(n0 + wcol, N - 1);
    const int wk = 8 * (tid / TN);
    if constexpr (SWIGLU) {  // (32 columns of gate, the same of up, and so on: 128 bytes of a row together)
      const int up = wcol >> 5 & 1, h = (wcol >> 6) * 32 + (wcol & 31);
      w_from = up * (N / 2) + min(n0 / 2 + h, N / 2 - 1);
      wcol = 2 * h + up;
    }
    const int x_unit = (xk >> 3) * S::kOctX + xrow;
    const int w_unit = 3 * S::kPartX + (wk >> 3) * S::kOctW + wcol / (32 * NB) * (36 * NB) + wcol % NB * 36 + wcol % (32 * NB) / NB;
    // fragments
    const int a_unit = j * S::kOctX + wm * 32 * MB + ln;
    const int b_unit = 3 * S::kPartX + j * S::kOctW + wn * 36 * NB + ln;

    // (rows past the last one repeat it and columns likewise: their products are never stored)
    const unsigned x_off = (unsigned)(((long long)min(m0 + xrow, T - 1) * g.xs + xk) * 4);
    const unsigned w_off = (unsigned)(((long long)wk * N + w_from) * 4);
    const char *x_base = (const char *)(g.x + k_begin);
    const char *w_base = (const char *)(g.w + (long long)k_begin * N);

    // two register sets: the tiles of step t travel in set t & 1 and are requested two steps ahead
    f32x4 sx[kSets][NX];
    float sw[kSets][8];
    int k_next = k_begin, to_load = nk;
    auto load_tiles = [&](f32x4 (&rx)[NX], float (&rw)[8]) {
#pragma unroll
      for (int u = 0; u < NX; ++u) {
        const int kk = k_next + xk + 4 * u;
        rx[u] = GUARD && kk >= k_end ? f32x4{0.f, 0.f, 0.f, 0.f} : *(const f32x4 *)(x_base + x_off + 16 * u);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float *row = (const float *)(w_base + (long long)i * N * 4);
        rw[i] = GUARD && k_next + wk + i >= k_end ? 0.f : *(const float *)((const char *)row + w_off);
      }
      if (--to_load > 0) {  // (behind the last step its tiles are requested again: the loop has no conditions)
        x_base += TK * 4;
        w_base += w_step;
        k_next += TK;
      }
    };
    auto park_tiles = [&](const f32x4 (&rx)[NX], const float (&rw)[8], u32x4 *stage) {
      u32x4 h, m, l;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        unsigned a, b, c;
        split_pair(rw[2 * i] * kLift, rw[2 * i + 1] * kLift, a, b, c);
        h[i] = a, m[i] = b, l[i] = c;
      }
      stage[w_unit] = h;
      stage[w_unit + S::kPartW] = m;
      stage[w_unit + 2 * S::kPartW] = l;
      if constexpr (NX == 1) {
        u32x2 *half = (u32x2 *)(stage + x_unit) + ((xk >> 2) & 1);
        split_quad(rx[0] * kLift, half[0], half[2 * S::kPartX], half[4 * S::kPartX]);
      } else {
        split_octet(rx[0] * kLift, rx[1] * kLift, h, m, l);
        stage[x_unit] = h;
        stage[x_unit + S::kPartX] = m;
        stage[x_unit + 2 * S::kPartX] = l;
      }
    };

    f32x16 acc[MB][NB];
#pragma unroll
    for (int a = 0; a < MB; ++a)
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;

    // (after the last barrier of the tile before this one nobody reads LDS any more)
    load_tiles(sx[0], sw[0]);
    if (kSets == 2) load_tiles(sx[kSets - 1], sw[kSets - 1]);
    park_tiles(sx[0], sw[0], lds[0]);
    load_tiles(sx[0], sw[0]);
    __syncthreads();

    // (smallest products first; the blocks take turns, no MFMA waits for the one before it)
    // Per step of 16 along K: the fragments are fetched, the next step's tiles are split and go to the other
    // stage while the MFMAs run, the tiles of a later step are requested into the registers just freed, one barrier.
    auto step = [&](const int kt, f32x4 (&rx)[NX], float (&rw)[8]) {  // rx, rw: the set that holds step kt + 1
      const u32x4 *stage = lds[kt & 1];
      u32x4 af[3][MB], bf[3][NB];
#pragma unroll
      for (int p = 0; p < 3; ++p) {
#pragma unroll
        for (int a = 0; a < MB; ++a) af[p][a] = stage[a_unit + p * S::kPartX + 32 * a];
#pragma unroll
        for (int b = 0; b < NB; ++b) bf[p][b] = stage[b_unit + p * S::kPartW + 36 * b];
      }
      park_tiles(rx, rw, lds[(kt & 1) ^ 1]);
      load_tiles(rx, rw);
#pragma unroll
      for (int p = 0; p < 6; ++p)
#pragma unroll
        for (int a = 0; a < MB; ++a)
#pragma unroll
          for (int b = 0; b < NB; ++b) acc[a][b] = mfma_bf16(af[kPartA[p]][a], bf[kPartB[p]][b], acc[a][b]);
      __syncthreads();
    };
    for (int kt = 0; kt < nk; kt += 2) {
      step(kt, sx[kSets - 1], sw[kSets - 1]);
      if (kt + 1 < nk) step(kt + 1, sx[0], sw[0]);
    }

    const int row0 = m0 + wm * 32 * MB + 4 * j, col = n0 + wn * 32 * NB + NB * ln;
    // sums that are not finite come from operands that are not (or overflow): again in fp32, which says which (2048 rows
    // of 2048 -> 16384 with one NaN in x: 1.3 ms against 0.65 without; one k at a time it was 13.9)
    float probe = 0.f, down = kDrop;
#pragma unroll
    for (int a = 0; a < MB; ++a)
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) probe = fmaf(acc[a][b][r], 0.f, probe);
    if (__any(probe != 0.f)) {
#pragma unroll
      for (int a = 0; a < MB; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;
      // eight k a turn, four of them a lane half's (K is a multiple of 4: those behind its end are zeros on both sides)
#pragma clang loop unroll(disable)
      for (int k0 = k_begin; k0 < k_end; k0 += 8) {
        const int k = k0 + 4 * j;
        const bool in = k < k_end;
        f32x4 xv[MB];
        typedef float Columns __attribute__((ext_vector_type(NB)));
        Columns wv[4];
#pragma unroll
        for (int a = 0; a < MB; ++a)
          xv[a] = in ? *(const f32x4 *)(g.x + (long long)min(m0 + (wm * MB + a) * 32 + ln, T - 1) * g.xs + k) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (SWIGLU) {
            const float *gate = g.w + (long long)(k + i) * N + min(col / 2, N / 2 - 1);
#pragma unroll
            for (int b = 0; b < NB; ++b) wv[i][b] = in ? gate[b * (N / 2)] : 0.f;
          } else {
            wv[i] = in ? *(const Columns *)(g.w + (long long)(k + i) * N + min(col, N - NB)) : Columns(0.f);
          }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int a = 0; a < MB; ++a)
#pragma unroll
            for (int b = 0; b < NB; ++b) acc[a][b] = mfma_f32(xv[a][i], wv[i][b], acc[a][b]);
      }
      down = 1.f;
    }

    // A piece travels as [pair of rows][thread] float4: consecutive threads, consecutive 16 bytes.
    constexpr long long kSlot = (long long)TM * TN;
    constexpr int kOut = 4 * MB * NB;
    f32x4 out[kOut];
#pragma unroll
    for (int a = 0; a < MB; ++a)
#pragma unroll
      for (int r = 0; r < 4 * NB; ++r)
        out[8 * a + r] = f32x4{acc[a][0][2 * r], acc[a][1][2 * r], acc[a][0][2 * r + 1], acc[a][1][2 * r + 1]} * down;
    const int in_slot = 4 * tid;
    if (g.pieces) {  // the second kernel adds the pieces
      float *slot = g.partials + blockIdx.x * kSlot + in_slot;
#pragma unroll
      for (int r = 0; r < kOut; ++r) *(f32x4 *)(slot + r * 4 * NT) = out[r];
      return;
    }
    if (s_end < steps) {
      leave_piece(g, g.partials + blockIdx.x * kSlot + in_slot, 4 * NT, out);
      continue;
    }
    if (s_begin > 0) {  // the tile's earlier pieces lie with the places before this one, from the one that holds the tile's first unit on
      const int p_first = t * steps / g.quota;
      add_earlier_pieces(g, group, p_first, place - p_first, kSlot, in_slot, 4 * NT, out);
    }
    if (col < N) {  // N is a multiple of 4: a lane's columns are inside together
#pragma unroll
      for (int r = 0; r < kOut; ++r) {
        if constexpr (SWIGLU)
          store_swiglu(g, row0, col / 2, r, out[r]);
        else
          store_four<NB>(g, row0, col, r, out[r]);
      }
    }
  }
}

// W of one part in tiles of 256 x 256 (WM 4: wavefronts of 64 rows and 128 columns) and 128 x 256 (WM 2: 64 x 64), on
// v_mfma_f32_16x16x32_bf16.  A step is 32 of K.  Stages of LDS: unit [part][octet of k][row] and [octet][block of 16 columns][place], as
// above but for 16 rows and 16 columns a block; column c of a wavefront's lies in block c % NB at place c / NB, so that a lane holds NB
// neighbouring columns of four rows of each block.
// The three products of a block follow each other on one accumulator.  What that is worth is power: a loop of nothing but these MFMAs reaches
// 2150 TFLOP/s on random numbers in this order, 2020 with the products outermost, and 1780 with v_mfma_f32_32x32x16_bf16 in any order.
// A wavefront holds the fragments of its columns of W for a step; those of its rows arrive one block of 16 ahead.  The next step's tiles are
// split and put into the other stage, and the registers asked for again at once, in small pieces of work behind each MFMA.
// Us, tiles of 32 x 32 blocks and steps of 16 | this, both launches where there are two: 2048 rows of 2048 -> 16384 344 | 318, 8192 -> 2048 185 | 167, 2048 -> 2048
// 60.6 | 57.1, 777 rows of 2048 -> 16384 164 | 144, 512 rows 90.9 | 85.4, of 8192 -> 2048 57.6 | 56.7, of 2048 -> 3072 30.6 | 30.6; with all loads, splits
// and writes of a step in its first half 325, 173, 59.7, 153, 90.7, 58.9.  Errors against 64 bits 0.3 to 2 % smaller (fewer roundings).
// PLANES: x comes as its parts, which go from memory to LDS by themselves (a row's 64 bytes of a step, the four octets of row r at places o ^ (r / 2 % 4),
// so that eight rows of an octet lie on eight banks' widths): no splits, a quarter of the writes.  The same bits.  Us, x | its parts: 2048 rows of
// 2048 -> 16384 320 | 298, 777 rows 149 | 131, 512 rows 93 | 83, 300 rows 82 | 76, 512 rows of 2048 -> 3072 32.4 | 30.6, 2048 rows of 2048 -> 2048 58 | 55,
// 8192 -> 2048 173 | 160, 512 rows 57 | 58.  The copies are not counted by the compiler: a step ends with a wait for all but its loads of W,
// which are requested behind them.
// Registers: tiles of 128 x 256 keep all, those of 256 x 256 spill 72 to 89 of a lane's (292 to 348 bytes of scratch), addresses and what a tile begins and ends with: none of it
// in the block that holds the MFMAs.
// What bounds it: on zeros 2048 rows of 2048 -> 16384 (x itself) take 279 us, of which the MFMAs and fragments are 201, splits 26, writes to LDS 31 (17
// cycles each while MFMAs run) and loads 21; on random numbers the clock is at 2.06 GHz.
// END: K ends with a step (kWhole; PLANES always); within one (kShifted): the last step is moved back until it ends with K, and what the steps before it
// have had of x counts as zeros, so that no load hangs on a condition; or within the only one (kGuarded).  Us, every load behind a condition | this:
// 512 rows of 2064 -> 16384 141 | 126, 777 rows of 1040 -> 16384 103 | 95, 1100 rows of 4112 -> 1028 58.5 | 49.8, 2048 rows of 2064 -> 2048 78.5 | 66.5, 8208 -> 2048
// 193 | 171, 512 rows of 2060 -> 16384 130 | 116, 1300 rows of 36 -> 16380 41.4 | 28.4.
constexpr int kWhole = 0, kShifted = 1, kGuarded = 2;
template <int WM, int END, bool SWIGLU, bool PLANES>
__global__ __launch_bounds__(512, 2) void sgemm_wide_kernel(const GemmArgs g) {
  constexpr int WN = 8 / WM, MB = 4, NB = 2 * WM, TM = 64 * WM, TN = 256, NT = 512;
  constexpr bool GUARD = END == kGuarded;
  static_assert(END == kWhole || !PLANES, "planes hold whole steps");
  constexpr int NX = WM / 2;               // octets of x a thread stages (of W: two); PLANES: 16 rows of a part that a wavefront copies
  constexpr int kSets = WM == 4 ? 1 : 2;   // register sets: tiles are requested one step (of 3072 cycles) ahead, or two (of 1536)
  // units of 16 bytes; blocks of W a few units apart from 16, so that eight neighbouring threads' columns lie on eight different ones modulo 8
  constexpr int kOctX = TM, kPartX = 4 * kOctX, kBlockW = NB == 8 ? (SWIGLU ? 18 : 17) : (SWIGLU ? 20 : 18), kOctW = WN * NB * kBlockW;
  constexpr int kW = 3 * kPartX, kUnits = kW + 4 * kOctW;
  __shared__ __attribute__((aligned(16))) u32x4 lds[2 * kUnits];

  // (workgroups and their runs as above)
  const int group = blockIdx.x & ((1 << g.group_bits) - 1), place = blockIdx.x >> g.group_bits;
  const int steps = g.steps;
  int u0 = place * g.quota, u1 = min(u0 + g.quota, g.tiles_per_group * steps);
  if (g.pieces) {
    const int t = place / g.pieces;
    u0 = t * steps + (place - t * g.pieces) * g.quota;
    u1 = t < g.tiles_per_group ? min(u0 + g.quota, (t + 1) * steps) : u0;
  }
  if (u0 >= u1) return;
  const int t_first = u0 / steps, t_last = (u1 - 1) / steps;
  const bool leaves_piece = u1 < (t_last + 1) * steps;

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int T = g.T, K = g.K, N = g.N;

  for (int visit = 0; visit <= t_last - t_first; ++visit) {
    const int t = leaves_piece ? (visit == 0 ? t_last : t_first + visit - 1) : t_first + visit;
    const int s_begin = t == t_first ? u0 - t_first * steps : 0;
    const int s_end = t == t_last ? u1 - t_last * steps : steps;
    const int tile = group * g.tiles_per_group + t;
    const int tm = tile % g.tiles_m, tn = tile / g.tiles_m;
    const int m0 = tm * TM, n0 = tn * TN;
    const int k_begin = s_begin * kWideStep, k_end = min(K, s_end * kWideStep);
    const int nk = s_end - s_begin;
    const int had = END == kShifted && s_end == steps ? steps * kWideStep - K : 0;  // of the last step's k

    int tid = threadIdx.x;  // (worked out again per tile, as above)
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63, ln = lane & 15, j = lane >> 4;

    // staging: x: octet tid / 8 % 4 of row tid % 8 + 8 (tid / 32) (and 128 on); W: octets tid / 256 and two on of column tid % 256
    const int xrow = (tid & 7) + 8 * (tid >> 5), xk = 8 * (tid >> 3 & 3);
    const int wk = 8 * (tid >> 8);
    int wcol = tid & 255, w_from = min(n0 + wcol, N - 1);
    if constexpr (SWIGLU) {  // (32 columns of gate, the same of up, and so on: 128 bytes of a row together; a lane holds both of a hidden column)
      const int up = wcol >> 5 & 1, h = (wcol >> 6) * 32 + (wcol & 31);
      w_from = up * (N / 2) + min(n0 / 2 + h, N / 2 - 1);
      wcol = NB * (h / (NB / 2)) + h % (NB / 2) + NB / 2 * up;
    }
    const int x_unit = (xk >> 3) * kOctX + xrow;
    const int w_unit = kW + (wk >> 3) * kOctW + wcol / (16 * NB) * (NB * kBlockW) + wcol % NB * kBlockW + wcol % (16 * NB) / NB;
    // fragments
    const int a_unit = PLANES ? (wm * 64 + ln) * 4 + (j ^ (ln >> 1 & 3)) : j * kOctX + wm * 64 + ln, b_unit = kW + j * kOctW + wn * (NB * kBlockW) + ln;

    // (rows past the last one repeat it and columns likewise: their products are never stored)
    unsigned x_off[NX], w_row[8];
#pragma unroll
    for (int u = 0; u < NX; ++u) {
      if constexpr (PLANES)
        x_off[u] = 64u * (unsigned)min(m0 + 16 * (wave + 8 * u) + (lane >> 2), T - 1) + 16u * ((lane & 3) ^ (lane >> 3 & 3));
      else
        x_off[u] = (unsigned)(((long long)min(m0 + xrow + 128 * u, T - 1) * g.xs + xk) * 4);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) w_row[i] = (unsigned)(((long long)(wk + i) * N + w_from) * 4);
    const int k_first = k_begin - (nk == 1 ? had : 0);
    const char *x_base = PLANES ? (const char *)(g.planes + (long long)k_begin * T) : (const char *)(g.x + k_first), *w_base = (const char *)(g.w + (long long)k_first * N);
    const long long plane = 2LL * T * K;

    f32x4 sx[kSets][NX][2];
    float sw[kSets][2][8];
    int k_next = k_begin, to_load = nk, to_copy = nk, to_split = nk;
    float lift[2];  // (kShifted) of an octet's halves
    auto set_lift = [&]() {
#pragma unroll
      for (int h = 0; h < 2; ++h) lift[h] = to_split == 1 && xk + 4 * h < had ? 0.f : kLift;
    };
    if constexpr (END == kShifted) set_lift();
    auto load_x = [&](const int set, const int u, const int h) {
      if constexpr (!PLANES) sx[set][u][h] = GUARD && k_next + xk + 4 * h >= k_end ? f32x4{0.f, 0.f, 0.f, 0.f} : load_from((const f32x4 *)(x_base + 16 * h), x_off[u]);
    };
    auto load_w = [&](const int set, const int o, const int i) {
      sw[set][o][i] = GUARD && k_next + wk + 16 * o + i >= k_end ? 0.f : load_from((const float *)(w_base + o * (64LL * N)), w_row[i]);
    };
    auto advance = [&]() {
      if (--to_load > 0) {  // (behind the last step its tiles are requested again: the loop has no conditions)
        const int by = kWideStep - (to_load == 1 ? had : 0);
        if constexpr (!PLANES) x_base += by * 4;
        w_base += (long long)by * N * 4;
        k_next += kWideStep;
      }
    };

    // The work beside the MFMAs, in pieces of at most four vector instructions (a SIMD issues two of them during an MFMA for nothing) or a write, of
    // which four wavefronts' take 70 cycles.  Per octet of x: four pairs split in four pieces each, three writes, two loads of the next; per octet of W: four
    // pairs, a write, eight loads.
    constexpr int kItemsX = PLANES ? 3 * NX : 21 * NX, kItems = kItemsX + 26;
    u32x4 whole[3];
    float pa, pb;
    auto item = [&](const int it, const int set, u32x4 *stage) {
      if (PLANES && it < kItemsX) {
        const int u = it / 3, p = it % 3;
        copy_to_lds<false>(stage + p * kPartX + 64 * (wave + 8 * u), x_base + p * plane, x_off[u]);
        if (it == kItemsX - 1 && --to_copy > 0) x_base += 64LL * T;
      } else if (it < kItemsX) {
        const int u = it / 21, m = it % 21, i = m / 4;
        if (m >= 19) {
          load_x(set, u, m - 19);
        } else if (m >= 16) {
          stage[x_unit + 128 * u + (m - 16) * kPartX] = whole[m - 16];
        } else if (m % 4 == 0) {
          pa = sx[set][u][i / 2][i % 2 * 2] * (END == kShifted ? lift[i / 2] : kLift);
          pb = sx[set][u][i / 2][i % 2 * 2 + 1] * (END == kShifted ? lift[i / 2] : kLift);
          whole[0][i] = pack_bf16(pa, pb);
        } else if (m % 4 == 1) {
          pa -= __builtin_bit_cast(float, whole[0][i] << 16);
          pb -= __builtin_bit_cast(float, whole[0][i] & 0xffff0000u);
        } else if (m % 4 == 2) {
          whole[1][i] = pack_bf16(pa, pb);
          pa -= __builtin_bit_cast(float, whole[1][i] << 16);
        } else {
          pb -= __builtin_bit_cast(float, whole[1][i] & 0xffff0000u);
          whole[2][i] = pack_bf16(pa, pb);
        }
      } else {
        const int o = (it - kItemsX) / 13, m = (it - kItemsX) % 13;
        if (m >= 5)
          load_w(set, o, m - 5);
        else if (m == 4)
          stage[w_unit + 2 * o * kOctW] = whole[0];
        else
          whole[0][m] = pack_high(sw[set][o][2 * m] * kLift, sw[set][o][2 * m + 1] * kLift);
      }
      if (it == kItems - 1) {
        advance();
        if constexpr (END == kShifted) --to_split, set_lift();
      }
    };
    auto load_all = [&](const int set) {
#pragma unroll
      for (int u = 0; u < (PLANES ? 0 : NX); ++u) load_x(set, u, 0), load_x(set, u, 1);
#pragma unroll
      for (int i = 0; i < 16; ++i) load_w(set, i / 8, i % 8);
      advance();
    };

    f32x4 acc[MB][NB];
#pragma unroll
    for (int a = 0; a < MB; ++a)
#pragma unroll
      for (int b = 0; b < NB; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x4 af[2][3], bf[NB];
    auto fetch_x = [&](const u32x4 *stage, const int a, const int p) { af[a & 1][p] = stage[a_unit + (PLANES ? 64 : 16) * a + p * kPartX]; };
    auto fetch_w = [&](const u32x4 *stage, const int b) { bf[b] = stage[b_unit + b * kBlockW]; };
    auto multiply = [&](const int a, const int b, const int p) { acc[a][b] = mfma_bf16_16(af[a & 1][p], bf[b], acc[a][b]); };

    // (after the last barrier of the tile before this one nobody reads what he uses any more)
    load_all(0);
    if constexpr (kSets == 2) load_all(1);
#pragma unroll
    for (int it = 0; it < kItems; ++it) item(it, 0, lds);
#pragma unroll
    for (int b = 0; b < NB; ++b) bf[b] = u32x4{0, 0, 0, 0};
#pragma unroll
    for (int p = 0; p < 3; ++p) af[(MB - 1) & 1][p] = u32x4{0, 0, 0, 0};
    if constexpr (PLANES) __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();

    // A turn of the loop is the last blocks of rows of the step before (of zeros in front of the first), in which the fragments of W and of the
    // first block of rows arrive, and all others of step kt.  (So the barrier stands where a turn ends: there the compiler waits for all of LDS anyway.)
    auto step = [&](const int kt, const int set) {  // set: holds the tiles of step kt + 1
      const u32x4 *const stage = lds + (kt & 1) * kUnits;
      u32x4 *const next = lds + ((kt & 1) ^ 1) * kUnits;
      constexpr int kSlots = 3 * MB * NB;
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        const int a = (i + MB - 1) % MB;
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int p = 2; p >= 0; --p) {  // smallest products first
            multiply(a, b, p);
            if (i == 0 && p == 0) fetch_w(stage, b);
            if (p == 1 && b < 3) fetch_x(stage, (a + 1) % MB, 2 - b);
            const int slot = 3 * (i * NB + b) + 2 - p;
#pragma unroll
            for (int it = slot * kItems / kSlots; it < (slot + 1) * kItems / kSlots; ++it) item(it, set, next);
            __builtin_amdgcn_sched_barrier(0);
          }
      }
      if constexpr (PLANES) __builtin_amdgcn_s_waitcnt(0x4F70);  // vmcnt(16): all but this step's loads of W, which were requested behind its copies
      __syncthreads();
    };
    if constexpr (kSets == 1) {
      for (int kt = 0; kt < nk; ++kt) step(kt, 0);
    } else {
      // (in pairs: a way out between them has the compiler wait for loads of the step before)
      for (int kt = 1; kt < nk; kt += 2) {
        step(kt - 1, 1);
        step(kt, 0);
      }
      if (nk & 1) step(nk - 1, 1);
    }
#pragma unroll
    for (int slot = 0; slot < 3 * NB; ++slot) multiply(MB - 1, slot / 3, 2 - slot % 3);

    const int row0 = m0 + wm * 64 + 4 * j, col = n0 + wn * 16 * NB + NB * ln;
    // sums that are not finite come from operands that are not (or overflow): again in fp32, which says which
    float probe = 0.f, down = kDrop;
#pragma unroll
    for (int a = 0; a < MB; ++a)
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) probe = fmaf(acc[a][b][r], 0.f, probe);
    if (__any(probe != 0.f)) {
#pragma unroll
      for (int a = 0; a < MB; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
      // 16 k a turn, four of them a quarter's (K is a multiple of 4: those behind its end are zeros on both sides)
#pragma clang loop unroll(disable)
      for (int k0 = k_begin; k0 < k_end; k0 += 16) {
        const int k = k0 + 4 * j;
        const bool in = k < k_end;
        f32x4 xv[MB];
#pragma unroll
        for (int a = 0; a < MB; ++a)
          xv[a] = !in      ? f32x4{0.f, 0.f, 0.f, 0.f}
                  : PLANES ? join_planes(g.planes + ((long long)(k / 32) * T + min(m0 + wm * 64 + 16 * a + ln, T - 1)) * 32 + k % 32, (long long)T * K)
                           : *(const f32x4 *)(g.x + (long long)min(m0 + wm * 64 + 16 * a + ln, T - 1) * g.xs + k);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int b = 0; b < NB; ++b) {
            const int from = SWIGLU ? b / (NB / 2) * (N / 2) + min(col / 2 + b % (NB / 2), N / 2 - 1) : min(col + b, N - 1);
            const float wv = in ? g.w[(long long)(k + i) * N + from] : 0.f;
#pragma unroll
            for (int a = 0; a < MB; ++a) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[a][i], wv, acc[a][b], 0, 0, 0);
          }
      }
      down = 1.f;
    }

    // A piece travels as [row of a block, four columns][thread] float4: consecutive threads, consecutive 16 bytes.
    constexpr long long kSlot = (long long)TM * TN;
    constexpr int Q = NB / 4, kOut = 4 * MB * Q;
    f32x4 out[kOut];
#pragma unroll
    for (int a = 0; a < MB; ++a)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int q = 0; q < Q; ++q)
          out[(4 * a + r) * Q + q] = f32x4{acc[a][4 * q][r], acc[a][4 * q + 1][r], acc[a][4 * q + 2][r], acc[a][4 * q + 3][r]} * down;
    const int in_slot = 4 * tid;
    if (g.pieces) {  // the second kernel adds the pieces
      float *slot = g.partials + blockIdx.x * kSlot + in_slot;
#pragma unroll
      for (int r = 0; r < kOut; ++r) *(f32x4 *)(slot + r * 4 * NT) = out[r];
      return;
    }
    if (s_end < steps) {
      leave_piece(g, g.partials + blockIdx.x * kSlot + in_slot, 4 * NT, out);
      continue;
    }
    if (s_begin > 0) {
      const int p_first = t * steps / g.quota;
      add_earlier_pieces(g, group, p_first, place - p_first, kSlot, in_slot, 4 * NT, out);
    }
#pragma unroll
    for (int a = 0; a < MB; ++a)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const f32x4 *const v = out + (4 * a + r) * Q;
        const int row = row0 + 16 * a + r;
        if constexpr (SWIGLU) {  // (N / 2 is a multiple of 4: a lane's hidden columns are inside together)
          if (row >= T || col >= N) continue;
          float *const y = g.y + (long long)row * (N / 2) + col / 2;
          if constexpr (Q == 1)
            *(f32x2 *)y = f32x2{swiglu(v[0].x, v[0].z), swiglu(v[0].y, v[0].w)};
          else
            *(f32x4 *)y = f32x4{swiglu(v[0].x, v[1].x), swiglu(v[0].y, v[1].y), swiglu(v[0].z, v[1].z), swiglu(v[0].w, v[1].w)};
        } else {
#pragma unroll
          for (int q = 0; q < Q; ++q)  // (N is a multiple of 4, not of a lane's columns)
            if (col + 4 * q < N) store_four<4>(g, row, col + 4 * q, 0, v[q]);
        }
      }
  }
}

// Few rows: a wavefront owns the columns of W it multiplies, so they go from memory to its registers and are split
// there; only x goes through LDS.  A workgroup of four wavefronts owns 32 rows and 128 columns and walks K in steps of 32:
// wavefronts 0 and 1 take the first half of a step, 2 and 3 the second, 64 columns each, and the two halves' sums meet in
// LDS at the end.  Lane n of a wavefront loads two neighbouring columns (a row of W 256 bytes at a time) and 8 rows, which
// are its fragments of two blocks.
// Against tiles of 64 x 128 with both operands in LDS, which this reads and writes a fifth as much (us): 32 rows of
// 2048 -> 16384 44 -> 30 (134 MB: 22 at the rate of a read), 2048 -> 3072 19.3 -> 14.4, 45 rows 44 -> 41 and 19.5 -> 15.7,
// 64 rows of 1024 -> 1024 12.1 -> 9.2.  64 rows by 128 columns this way were slower than 32 (45 rows of
// 8192 -> 2048 34 against 30.5).  Bound by a launch, the first loads and the kernel that adds the pieces where the
// weights are small, by reading them where they are not.
template <bool GUARD>
__global__ __launch_bounds__(256, 2) void sgemm_few_kernel(const GemmArgs g) {
  constexpr int TM = 32, TN = 128, TS = kFewStep;
  constexpr int kOct = TM + 4, kPart = 4 * kOct;  // units of 16 bytes: four octets of k, four units apart from a multiple of 16
  constexpr int kStage = 3 * kPart;
  constexpr int kMerge = 2 * 2 * 16 * 64 / 4;  // units that two wavefronts' sums take
  __shared__ __attribute__((aligned(16))) u32x4 lds[2 * kStage > kMerge ? 2 * kStage : kMerge];

  const int group = blockIdx.x & ((1 << g.group_bits) - 1), place = blockIdx.x >> g.group_bits;
  const int steps = g.steps, pieces = g.pieces ? g.pieces : 1;
  const int t = place / pieces, s_begin = (place - t * pieces) * g.quota, s_end = min(s_begin + g.quota, steps);
  if (t >= g.tiles_per_group || s_begin >= s_end) return;
  const int tile = group * g.tiles_per_group + t;
  const int m0 = tile % g.tiles_m * TM, n0 = tile / g.tiles_m * TN;
  const int T = g.T, K = g.K, N = g.N;
  const int k_begin = s_begin * TS, k_end = min(K, s_end * TS), nk = s_end - s_begin;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ln = lane & 31, j = lane >> 5, wn = wave & 1, kg = wave >> 1;
  const int col = n0 + 64 * wn + 2 * ln;

  // x: a thread takes four k, piece tid % 8, of row tid / 8 (rows past the last one repeat it)
  const int xrow = threadIdx.x >> 3, xk = 4 * (threadIdx.x & 7);
  const unsigned x_off = (unsigned)(((long long)min(m0 + xrow, T - 1) * g.xs + xk) * 4);
  u32x2 *const x_lds = (u32x2 *)(lds + (xk >> 3) * kOct + xrow) + (xk >> 2 & 1);
  // W: rows 16 kg + 8 j .. + 7 of a step (columns past the last two repeat them)
  const int wk = 16 * kg + 8 * j;
  const unsigned w_off = (unsigned)(((long long)wk * N + min(col, N - 2)) * 4);
  const char *x_base = (const char *)(g.x + k_begin), *w_base = (const char *)(g.w + (long long)k_begin * N);
  const long long row_bytes = 4LL * N;

  // register sets: the tiles of step t travel in set t & 1 and are requested two steps ahead (behind the last step
  // its tiles are requested again: the loop has no conditions)
  f32x4 sx[2];
  f32x2 sw[2][8];
  int k_next = k_begin, to_load = nk;
  auto load_tiles = [&](int set) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      sw[set][i] = !GUARD || k_next + wk + i < k_end ? *(const f32x2 *)(w_base + i * row_bytes + w_off) : f32x2{0.f, 0.f};
    sx[set] = !GUARD || k_next + xk < k_end ? *(const f32x4 *)(x_base + x_off) : f32x4{0.f, 0.f, 0.f, 0.f};
    if (--to_load > 0) {
      x_base += TS * 4;
      w_base += TS * row_bytes;
      k_next += TS;
    }
  };
  auto park_x = [&](int set, int stage) {
    u32x2 *at = x_lds + 2 * stage * kStage;
    split_quad(sx[set] * kLift, at[0], at[2 * kPart], at[4 * kPart]);
  };

  // The products of the first parts, and the others', 2^-8 of them: added up by themselves these round to next to
  // nothing.  Every 16 steps the first go to a sum of their own.  Five to sixteen rows came from the split GEMV, whose
  // sums are short: relative error of 17 rows in one accumulator | this way | the GEMV's, 1e-8: 1024 -> 1024 13.1 | 8.0 |
  // 9.0, 2048 -> 16384 24.4 | 10.2 | 12.4, 8192 -> 3072 26 | 12.1 | 12.8, 8192 -> 57344 103 | 12.1 | 21.5.
  f32x16 acc[2], rest[2], sum[2];
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[b][r] = rest[b][r] = sum[b][r] = 0.f;

  load_tiles(0);
  load_tiles(1);
  park_x(0, 0);
  __syncthreads();
  auto step = [&](const int kt, const int set) {  // set: holds step kt, the other one step kt + 1
    const u32x4 *stage = lds + (kt & 1) * kStage + (2 * kg + j) * kOct + ln;
    u32x4 af[3], bf[3][2];
#pragma unroll
    for (int p = 0; p < 3; ++p) af[p] = stage[p * kPart];
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        unsigned h, m, l;
        split_pair(sw[set][2 * i][b] * kLift, sw[set][2 * i + 1][b] * kLift, h, m, l);
        bf[0][b][i] = h, bf[1][b][i] = m, bf[2][b][i] = l;
      }
    park_x(set ^ 1, (kt & 1) ^ 1);
    load_tiles(set);
#pragma unroll
    for (int p = 0; p < 5; ++p)
#pragma unroll
      for (int b = 0; b < 2; ++b) rest[b] = mfma_bf16(af[kPartA[p]], bf[kPartB[p]][b], rest[b]);
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[b] = mfma_bf16(af[0], bf[0][b], acc[b]);
    __syncthreads();
  };
  for (int k0 = 0; k0 < nk; k0 += 16) {
    for (int kt = k0; kt < min(k0 + 16, nk); kt += 2) {
      step(kt, 0);
      if (kt + 1 < nk) step(kt + 1, 1);
    }
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) sum[b][r] += acc[b][r], acc[b][r] = 0.f;
  }

#pragma unroll
  for (int b = 0; b < 2; ++b) acc[b] = sum[b] + rest[b];
  const int row0 = m0 + 4 * j;
  // sums that are not finite come from operands that are not (or overflow): again in fp32, which says which
  float probe = 0.f;
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) probe = fmaf(acc[b][r], 0.f, probe);
  if (__any(probe != 0.f)) {
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[b][r] = 0.f;
#pragma clang loop unroll(disable)
    for (int k0 = k_begin + 16 * kg; k0 < k_end; k0 += (k0 & 15) ? 24 : 8) {  // (this wavefront's halves of the steps)
      const int k = k0 + 4 * j;
      const bool in = k < k_end;
      const f32x4 xv = in ? *(const f32x4 *)(g.x + (long long)min(m0 + ln, T - 1) * g.xs + k) : f32x4{0.f, 0.f, 0.f, 0.f};
      f32x2 wv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        wv[i] = in ? *(const f32x2 *)(g.w + (long long)(k + i) * N + min(col, N - 2)) : f32x2{0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[b] = mfma_f32(xv[i], wv[i][b], acc[b]);
    }
  } else {
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[b] *= kDrop;
  }
  // (every wavefront is past the last step's barrier: nobody reads tiles any more)
  f32x4 *const merge = (f32x4 *)lds + wn * (kMerge / 2) + lane;
  if (kg == 1) {
#pragma unroll
    for (int r = 0; r < 8; ++r) merge[64 * r] = f32x4{acc[0][2 * r], acc[1][2 * r], acc[0][2 * r + 1], acc[1][2 * r + 1]};
  }
  __syncthreads();
  if (kg == 1) return;
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const f32x4 v = f32x4{acc[0][2 * r], acc[1][2 * r], acc[0][2 * r + 1], acc[1][2 * r + 1]} + merge[64 * r];
    if (g.pieces) {  // [pair of rows][thread], as the kernel that adds the pieces takes them
      *(f32x4 *)(g.partials + (long long)blockIdx.x * (TM * TN) + r * 512 + 4 * threadIdx.x) = v;
    } else if (col < N) {
      const int row = row0 + 8 * (r >> 1) + 2 * (r & 1);
      store_pair(g, row, col, f32x2{v.x, v.y});
      store_pair(g, row + 1, col, f32x2{v.z, v.w});
    }
  }
}

// The same by weights of one part, which leaves registers for more rows: a workgroup of eight wavefronts owns 32 MB
// rows and 256 / KG columns, 32 of them a wavefront, and walks K in steps of 16 KG, of which each of KG groups of wavefronts
// takes its own 16.  W goes from memory to registers four steps ahead (64 KB in flight on a compute unit), x through LDS.
// Sums as in the kernel above, emptied every four steps, three products instead of six: no larger an error than
// that kernel's anywhere (1e-8, 17 rows: 1024 -> 1024 7.9 | 7.9, 2048 -> 16384 8.4 | 10.2, 8192 -> 2048 10.3 | 12.1; emptied every eight
// steps 96 rows of 768 -> 2304 7.9 | 7.6).
// Bound by reading W where it is large: nothing but these loads takes 24.9 us for 2048 -> 16384 and 17.9 for 8192 -> 2048, a launch
// of 4 included.  Loads of x that hung on a condition had the compiler wait for every load in flight once in four steps,
// and twice in front of the loop; and wavefronts that fetch fragments, split, multiply and meet, one after the other, all
// at the same time, leave each of these idle while the others last.  Us without the kernel that adds pieces, such loops | now: 45
// rows of 2048 -> 16384 30.7 | 27.0, 8192 -> 2048 24.1 | 21.9, 2048 -> 3072 12.5 | 10.6, 17 rows of 2048 -> 16384 30.1 | 26.4, 777 rows of
// 1024 -> 2048 24.8 | 21.8, 1024 -> 1024 15.1 | 13.6.  (Fragments a step ahead serve the 64-row tiles only: tiles of 32 rows have
// three MFMAs to put the rest between and are level or slower, 96 rows have no registers for them.  Tried and not kept:
// non-temporal loads of W, 30.7 | 32.7; eight wavefronts that take 64 columns and every eighth step by themselves, without a barrier:
// 32.9; tiles of 64 x 64: level at best.)
// SWIGLU (no pieces): wavefronts take 32 columns of gate and 32 of up in turn, and hand over by LDS.
template <int MB, int KG, bool GUARD, bool SWIGLU>
__global__ __launch_bounds__(512, 1) void sgemm_stream_kernel(const GemmArgs g) {
  constexpr bool AHEAD = MB == 2;  // whether fragments are fetched a step ahead
  constexpr int WN = 8 / KG, TM = 32 * MB, TN = 32 * WN, TS = 16 * KG, kSets = 4;
  constexpr int kOct = TM + 4, kPart = 2 * KG * kOct, kStage = 3 * kPart;  // units of 16 bytes, as above
  constexpr int kSums = MB * 16 * 64 / 4;                                  // units that a wavefront's sums take
  constexpr int kRows = 128 / KG, kRounds = (TM + kRows - 1) / kRows;      // rows that all threads stage at once
  __shared__ __attribute__((aligned(16))) u32x4 lds[2 * kStage > (8 - WN) * kSums ? 2 * kStage : (8 - WN) * kSums];

  const int group = blockIdx.x & ((1 << g.group_bits) - 1), place = blockIdx.x >> g.group_bits;
  const int steps = g.steps, pieces = g.pieces ? g.pieces : 1;
  const int t = place / pieces, s_begin = (place - t * pieces) * g.quota, s_end = min(s_begin + g.quota, steps);
  if (t >= g.tiles_per_group || s_begin >= s_end) return;
  const int tile = group * g.tiles_per_group + t;
  const int m0 = tile % g.tiles_m * TM, n0 = tile / g.tiles_m * TN;
  const int T = g.T, K = g.K, N = g.N;
  const int k_begin = s_begin * TS, k_end = min(K, s_end * TS), nk = s_end - s_begin;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ln = lane & 31, j = lane >> 5, wn = wave % WN, kg = wave / WN;
  const int col = SWIGLU ? n0 / 2 + 32 * (wn / 2) + ln : n0 + 32 * wn + ln, columns = SWIGLU ? N / 2 : N;
  const int w_from = min(col, columns - 1) + (SWIGLU ? wn % 2 * columns : 0);

  // x: a thread takes four k, piece tid % (4 KG), of row tid / (4 KG) (and kRows on; rows past the last one repeat it)
  const int xrow = threadIdx.x / (4 * KG), xk = 4 * (threadIdx.x % (4 * KG));
  unsigned x_off[kRounds];
#pragma unroll
  for (int u = 0; u < kRounds; ++u) x_off[u] = (unsigned)(((long long)min(m0 + xrow + kRows * u, T - 1) * g.xs + xk) * 4);
  u32x2 *const x_lds = (u32x2 *)(lds + (xk >> 3) * kOct + xrow) + (xk >> 2 & 1);
  // W: rows 16 kg + 8 j .. + 7 of a step (columns past the last one repeat it)
  const int wk = 16 * kg + 8 * j;
  const unsigned w_off = (unsigned)(((long long)(GUARD ? 0 : 8 * j) * N + w_from) * 4);
  const char *x_base = (const char *)(g.x + k_begin), *w_base = (const char *)(g.w + (long long)(k_begin + (GUARD ? 0 : 16 * kg)) * N);
  const long long row_bytes = 4LL * N;

  // Register sets: what step t takes of W travels in set t % 4 and is requested four or five steps ahead, its x likewise.  Behind
  // the end the last step's is requested again, x counts as zeros, and so it does where K ends within a step (GUARD): no load
  // hangs on a condition, in front of which the compiler would wait for all those in flight.
  f32x4 sx[kSets][kRounds];
  float sw[kSets][8];
  int x_step = 0, w_step = 0;  // to be requested next
  auto load_x = [&](const int set) {
#pragma unroll
    for (int u = 0; u < kRounds; ++u)
      sx[set][u] = load_at((const f32x4 *)x_base, GUARD && k_begin + x_step * TS + xk >= k_end ? x_off[u] - 4 * xk : x_off[u]);
    if (x_step + 1 < nk) {
      ++x_step;
      x_base += TS * 4;
    }
  };
  auto load_w = [&](const int set) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      sw[set][i] = GUARD ? load_at((const float *)w_base, (unsigned)(min(wk + i, k_end - k_begin - w_step * TS - 1) * row_bytes) + w_off)
                         : load_at((const float *)(w_base + i * row_bytes), w_off);
    if (w_step + 1 < nk) {
      ++w_step;
      w_base += TS * row_bytes;
    }
  };
  unsigned parts[kRounds][3][2];  // of x of step t
  auto split_x = [&](const int t, const int set) {
    const float lift = (GUARD ? k_begin + t * TS + xk < k_end : t < nk) ? kLift : 0.f;
#pragma unroll
    for (int u = 0; u < kRounds; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        split_pair(sx[set][u][2 * h] * lift, sx[set][u][2 * h + 1] * lift, parts[u][0][h], parts[u][1][h], parts[u][2][h]);
  };
  auto park_x = [&](const int stage) {
#pragma unroll
    for (int u = 0; u < kRounds; ++u) {
      if (TM % kRows != 0 && xrow + kRows * u >= TM) continue;
      u32x2 *at = x_lds + 2 * (stage * kStage + kRows * u);
#pragma unroll
      for (int p = 0; p < 3; ++p) at[2 * p * kPart] = u32x2{parts[u][p][0], parts[u][p][1]};
    }
  };

  f32x16 acc[MB], rest[MB], sum[MB];
#pragma unroll
  for (int a = 0; a < MB; ++a)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[a][r] = rest[a][r] = sum[a][r] = 0.f;

  auto empty = [&]() {
#pragma unroll
    for (int a = 0; a < MB; ++a)
#pragma unroll
      for (int r = 0; r < 16; ++r) sum[a][r] += acc[a][r], acc[a][r] = 0.f;
  };
  u32x4 af[AHEAD ? 2 : 1][3][MB], bf[AHEAD ? 2 : 1];
  auto fetch_x = [&](const int set, const int stage, const int p, const int a) {
    af[set][p][a] = lds[stage * kStage + (2 * kg + j) * kOct + ln + p * kPart + 32 * a];
  };
  auto pack_w = [&](const int set, const int from, const int i) { bf[set][i] = pack_high(sw[from][2 * i] * kLift, sw[from][2 * i + 1] * kLift); };
  auto multiply = [&](const int set, const int p, const int a) {  // smallest products first
    f32x16 &to = p ? rest[a] : acc[a];
    to = mfma_bf16(af[set][p][a], bf[set], to);
  };

  // (what is needed first is requested first)
  load_w(0);
  load_x(0);
  load_x(1);
#pragma unroll
  for (int set = 1; set < kSets; ++set) load_w(set);
  load_x(2);
  load_x(3);
  split_x(0, 0);
  park_x(0);
  load_x(0);
  if constexpr (!AHEAD) {
    __syncthreads();
    auto step = [&](const int t, const int at) {  // at: t % 4
#pragma unroll
      for (int i = 0; i < 4; ++i) pack_w(0, at, i);
#pragma unroll
      for (int i = 0; i < 3 * MB; ++i) fetch_x(0, at & 1, i / MB, i % MB);
      split_x(t + 1, (at + 1) % kSets);
      park_x((at & 1) ^ 1);
      load_x((at + 1) % kSets);
      load_w(at);
#pragma unroll
      for (int i = 0; i < 3 * MB; ++i) multiply(0, 2 - i / MB, i % MB);
      __syncthreads();
    };
    for (int t = 0; t < nk; t += 4) {
      step(t, 0);
      step(t + 1, 1);
      step(t + 2, 2);
      step(t + 3, 3);
      empty();
    }
  } else {
    // Fragments are fetched a step ahead, from the stage that is whole since the last barrier, and the x of the step behind that
    // one goes into the stage whose fragments everybody has.  What else a step does stands between its MFMAs: left to itself the
    // compiler puts it behind them, and all wavefronts are at the same of the two at the same time.
    split_x(1, 1);
    park_x(1);
    load_x(1);
#pragma unroll
    for (int i = 0; i < 4; ++i) pack_w(0, 0, i);
    load_w(0);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 3 * MB; ++i) fetch_x(0, 0, i / MB, i % MB);
    __syncthreads();
    auto step = [&](const int t, const int at) {  // at: t % 4
      const int cur = at & 1, next = cur ^ 1;
#pragma unroll
      for (int slot = 0; slot < 3 * MB; ++slot) {
        multiply(cur, 2 - slot / MB, slot % MB);
#pragma unroll
        for (int i = 2 * slot; i < 2 * slot + 2 && i < 3 * MB; ++i) fetch_x(next, next, 2 - i / MB, i % MB);
        if (slot < 2) {
          pack_w(next, (at + 1) % kSets, 2 * slot);
          pack_w(next, (at + 1) % kSets, 2 * slot + 1);
          if (slot == 1) load_w((at + 1) % kSets);
        } else if (slot == 2) {
          split_x(t + 2, (at + 2) % kSets);
          park_x(cur);
          load_x((at + 2) % kSets);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      __syncthreads();
    };
    for (int t = 0; t < nk; t += 4) {
      step(t, 0);
      step(t + 1, 1);
      step(t + 2, 2);
      step(t + 3, 3);
      empty();
    }
  }

#pragma unroll
  for (int a = 0; a < MB; ++a) acc[a] = sum[a] + rest[a];
  // sums that are not finite come from operands that are not (or overflow): again in fp32, which says which
  float probe = 0.f;
#pragma unroll
  for (int a = 0; a < MB; ++a)
#pragma unroll
    for (int r = 0; r < 16; ++r) probe = fmaf(acc[a][r], 0.f, probe);
  if (__any(probe != 0.f)) {
#pragma unroll
    for (int a = 0; a < MB; ++a)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[a][r] = 0.f;
#pragma clang loop unroll(disable)
    for (int k0 = k_begin + 16 * kg; k0 < k_end; k0 += (k0 & 15) ? TS - 8 : 8) {  // (this wavefront's part of the steps)
      const int k = k0 + 4 * j;
      const bool in = k < k_end;
      f32x4 xv[MB];
      float wv[4];
#pragma unroll
      for (int a = 0; a < MB; ++a)
        xv[a] = in ? *(const f32x4 *)(g.x + (long long)min(m0 + 32 * a + ln, T - 1) * g.xs + k) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; ++i) wv[i] = in ? g.w[(long long)(k + i) * N + w_from] : 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int a = 0; a < MB; ++a) acc[a] = mfma_f32(xv[a][i], wv[i], acc[a]);
    }
  } else {
#pragma unroll
    for (int a = 0; a < MB; ++a) acc[a] *= kDrop;
  }
  // (every wavefront is past the last step's barrier: nobody reads tiles any more)
  f32x4 *const merge = (f32x4 *)lds + wn * kSums + lane;
  if (kg > 0) {
#pragma unroll
    for (int a = 0; a < MB; ++a)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        merge[(kg - 1) * WN * kSums + 64 * (4 * a + r)] = f32x4{acc[a][4 * r], acc[a][4 * r + 1], acc[a][4 * r + 2], acc[a][4 * r + 3]};
  }
  __syncthreads();
  if (!SWIGLU && kg > 0) return;
#pragma unroll
  for (int a = 0; a < MB; ++a)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (SWIGLU && kg > 0) continue;
      f32x4 v = f32x4{acc[a][4 * r], acc[a][4 * r + 1], acc[a][4 * r + 2], acc[a][4 * r + 3]};
      const f32x4 *const other = merge + 64 * (4 * a + r);
      v += other[0];  // (in pairs: four groups' sums one after the other round a little more)
      if constexpr (KG == 4) v += other[WN * kSums] + other[2 * WN * kSums];
      if constexpr (SWIGLU) {  // (each lane puts what it has where it found the first other sum)
        merge[64 * (4 * a + r)] = v;
      } else if (g.pieces) {  // row by row
        float *const piece = g.partials + (long long)blockIdx.x * (TM * TN) + (32 * a + 8 * r + 4 * j) * TN + 32 * wn + ln;
#pragma unroll
        for (int i = 0; i < 4; ++i) piece[i * TN] = v[i];
      } else if (col < N) {
        store_four<1>(g, m0 + 4 * j, col, 4 * a + r, v);
      }
    }
  if constexpr (SWIGLU) {
    __syncthreads();
    // (all wavefronts: those of a pair of gate and up take its registers of four in turn)
    constexpr int kShare = 2 * KG;  // wavefronts that share a pair of the sums
    const int share = kg * 2 + wn % 2;
    const f32x4 *const gate = (const f32x4 *)lds + wn / 2 * 2 * kSums + lane, *const up = gate + kSums;
#pragma unroll
    for (int i = 0; i < (4 * MB + kShare - 1) / kShare; ++i) {
      const int at = share + kShare * i;
      if (at >= 4 * MB || col >= columns) continue;
      const f32x4 a = gate[64 * at], b = up[64 * at];
      const int row = m0 + 4 * j + row_of<1>(at);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float v = swiglu(a[e], b[e]);
        if (row + e < T) g.y[(long long)(row + e) * columns + col] = v;
      }
    }
  }
}

// acc + piece 0 + piece 1 + ..., all C in flight
template <int C>
__device__ __forceinline__ f32x4 add_pieces(f32x4 acc, const float *piece, long long step) {
  f32x4 v[C];
#pragma unroll
  for (int c = 0; c < C; ++c) v[c] = *(const f32x4 *)(piece + c * step);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int c = 0; c < C; ++c) acc += v[c];
  return acc;
}

// How a product's tiles lie in its workgroups' slots.  `columns` of a lane: 1: row by row; 2: [pair of rows][thread] float4, two
// neighbouring columns of two rows of blocks of 32; 4 and 8: [row, four columns][thread] float4, of blocks of 16 rows.
struct PieceShape {
  int tm, tn;      // rows and columns of a tile
  int rows, wn;    // rows of a wavefront, wavefronts along the columns
  int threads;     // of the workgroup
};

// Where the first piece of (row, col) lies: four columns of a row, or (COLUMNS 2) two columns of two rows.
template <int COLUMNS>
__device__ __forceinline__ const float *first_piece(const GemmArgs &g, const PieceShape &s, int row, int col) {
  const int tm = row / s.tm, tn = col / s.tn, r = row - tm * s.tm, c = col - tn * s.tn;
  const int tile = tn * g.tiles_m + tm, group = tile / g.tiles_per_group, t = tile - group * g.tiles_per_group;
  const float *slot = g.partials + (((long long)t * g.pieces << g.group_bits) | group) * s.tm * s.tn;
  if constexpr (COLUMNS == 1) return slot + r * s.tn + c;
  const int wm = r / s.rows, q = r - wm * s.rows;
  int out, thread;
  if constexpr (COLUMNS == 2) {
    const int in = q & 31, at = 4 * (in >> 3) + (in & 3);  // (of the 16 registers of a block)
    out = 8 * (q >> 5) + at / 2;
    thread = (wm * s.wn + c / 64) * 64 + 32 * (in >> 2 & 1) + c % 64 / 2;
  } else {
    out = (4 * (q >> 4) + (q & 3)) * (COLUMNS / 4) + c % COLUMNS / 4;
    thread = (wm * s.wn + c / (16 * COLUMNS)) * 64 + 16 * (q >> 2 & 3) + c % (16 * COLUMNS) / COLUMNS;
  }
  return slot + 4 * ((long long)out * s.threads + thread);
}

// piece 0 + piece 1 + ... in that order, four of them in flight: 16 pieces of 17 rows of 132 columns 5.4 us one after the other, 4.1
// two at a time, 3.6 so, 3.1 eight at a time; launches that fill the chip take the same time each way.  Only pieces
// that are there are requested, and nothing for rows that pad a tile: with them 777 rows of 8192 -> 4092 took 14.4 us, not 11.4.
__device__ __forceinline__ f32x4 sum_of_pieces(const GemmArgs &g, const PieceShape &s, const float *piece) {
  const long long step = (long long)s.tm * s.tn << g.group_bits;
  f32x4 acc = {-0.f, -0.f, -0.f, -0.f};  // (which adds nothing to anything)
  int left = min(g.pieces, (g.steps + g.quota - 1) / g.quota);  // pieces that hold any steps
  for (; left >= 4; left -= 4, piece += 4 * step) acc = add_pieces<4>(acc, piece, step);
  if (left == 3)
    acc = add_pieces<3>(acc, piece, step);
  else if (left == 2)
    acc = add_pieces<2>(acc, piece, step);
  else if (left == 1)
    acc = add_pieces<1>(acc, piece, step);
  return acc;
}

// y = (res +) the sum of a product's pieces, or (SWIGLU) silu(gate) * up of its columns gate | up.  A thread takes what a lane of
// the product held in one register of four: grid (columns, rows).
template <int COLUMNS, bool SWIGLU>
__global__ __launch_bounds__(256) void sgemm_sum_kernel(const GemmArgs g, const PieceShape s) {
  constexpr int R = COLUMNS == 2 ? 2 : 1, C = 4 / R;
  const int row = R * blockIdx.y, col = C * (blockIdx.x * blockDim.x + threadIdx.x), N = SWIGLU ? g.N / 2 : g.N;
  if (col >= N) return;
  const f32x4 v = sum_of_pieces(g, s, first_piece<COLUMNS>(g, s, row, col));
  if constexpr (SWIGLU) {
    const f32x4 u = sum_of_pieces(g, s, first_piece<COLUMNS>(g, s, row, N + col));
    const f32x4 h = {swiglu(v.x, u.x), swiglu(v.y, u.y), swiglu(v.z, u.z), swiglu(v.w, u.w)};
    float *y = g.y + (long long)row * N + col;
    if constexpr (R == 1) {
      *(f32x4 *)y = h;
    } else {
      *(f32x2 *)y = f32x2{h.x, h.y};
      if (row + 1 < g.T) *(f32x2 *)(y + N) = f32x2{h.z, h.w};
    }
  } else {
    store_four<R == 1 ? 4 : 2>(g, row, col, 0, v);
  }
}

// The sum is q | k | v heads: queries and keys are rotated (prep_math.hpp's arithmetic) and, with the values, put where the attention
// reads them.  A thread takes the same place of a head's two halves.  Bound by a launch and its round trips; us, a sum and the launch that
// rotates | this: 45 rows of 2048 -> 3072 4.1 + 3.3 | 4.6, 512 rows 7.5 + 5.3 | 8.1.
template <int COLUMNS>
__global__ __launch_bounds__(256) void sgemm_sum_prep_kernel(const GemmArgs g, const PieceShape s, const GemvPrep p) {
  constexpr int R = COLUMNS == 2 ? 2 : 1, C = 4 / R;
  const int half = p.hd / 2, per = half / C, heads = p.H + 2 * p.KV, item = blockIdx.x * 256 + threadIdx.x;
  if (item >= heads * per) return;
  const int head = item / per, i = C * (item - head * per), row = R * blockIdx.y, col = head * p.hd + i;
  const bool second = R == 2 && row + 1 < g.T;
  float2 cs[R][C];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int c = 0; c < C; ++c) cs[r][c] = p.rope_tab[(long long)(p.start_pos + min(row + r, g.T - 1)) * half + i + c];
  f32x4 a = sum_of_pieces(g, s, first_piece<COLUMNS>(g, s, row, col)), b = sum_of_pieces(g, s, first_piece<COLUMNS>(g, s, row, col + half));
  if (head < p.H + p.KV) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
#pragma clang fp contract(off)
      const float2 t = cs[e / C][e % C];
      const float p0 = a[e] * t.x, p1 = b[e] * t.y, p2 = b[e] * t.x, p3 = a[e] * t.y;
      a[e] = p0 - p1;
      b[e] = p2 + p3;
    }
  }
  const int kv = head < p.H + p.KV ? head - p.H : head - p.H - p.KV;
  float *const to = head < p.H ? p.q_rot + ((long long)row * p.H + head) * p.hd + i
                               : (head < p.H + p.KV ? p.kc : p.vc) + ((long long)kv * p.cap + p.start_pos + row) * p.hd + i;
  const long long next = head < p.H ? (long long)p.H * p.hd : p.hd;  // floats to the same place of the next row
  if constexpr (R == 1) {
    *(f32x4 *)to = a;
    *(f32x4 *)(to + half) = b;
  } else {
    *(f32x2 *)to = f32x2{a.x, a.y};
    *(f32x2 *)(to + half) = f32x2{b.x, b.y};
    if (second) {
      *(f32x2 *)(to + next) = f32x2{a.z, a.w};
      *(f32x2 *)(to + next + half) = f32x2{b.z, b.w};
    }
  }
}

// The same, and the norm of the whole rows, which the next product reads, in one launch: a workgroup takes a row (COLUMNS 2: two rows), a
// thread up to two registers of four.  The sums of squares are fp64, as rms_norm.cr has them.  Bound by a launch and two round trips; us, a
// sum and a norm | this: 45 rows of 8192 -> 2048, 16 pieces, 4.9 + 3.9 | 5.0, of 2048 -> 2048 3.9 + 4.2 | 4.3; 512 rows of 8192 -> 2048, 8
// pieces, 8.3 + 5.1 | 11.0, 2048 rows, 4 pieces, with Dynamic Tanh 18.6 + 7.2 | 24.5.
template <int COLUMNS>
__global__ __launch_bounds__(1024) void sgemm_sum_norm_kernel(const GemmArgs g, const PieceShape s, const NextNorm norm) {
  constexpr int R = COLUMNS == 2 ? 2 : 1, C = 4 / R, kMost = 2;
  __shared__ double red[R][16];
  const int row = R * blockIdx.x, N = g.N;
  const bool second = R == 2 && row + 1 < g.T;
  f32x4 v[kMost], res[kMost];
  double sq[R] = {};
#pragma unroll
  for (int u = 0; u < kMost; ++u) {  // (the residual is requested in front of the pieces, whose sums wait for theirs)
    const int col = C * (threadIdx.x + u * blockDim.x);
    res[u] = f32x4{-0.f, -0.f, -0.f, -0.f};
    if (!g.res || col >= N) continue;
    const float *at = g.res + (long long)row * N + col;
    if constexpr (R == 1) {
      res[u] = *(const f32x4 *)at;
    } else {
      const f32x2 a = *(const f32x2 *)at, b = *(const f32x2 *)(at + (second ? N : 0));
      res[u] = f32x4{a.x, a.y, b.x, b.y};
    }
  }
#pragma unroll
  for (int u = 0; u < kMost; ++u) {
    const int col = C * (threadIdx.x + u * blockDim.x);
    v[u] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (col >= N) continue;
    v[u] = res[u] + sum_of_pieces(g, s, first_piece<COLUMNS>(g, s, row, col));
    float *at = g.y + (long long)row * N + col;
    if constexpr (R == 1) {
      *(f32x4 *)at = v[u];
    } else {
      *(f32x2 *)at = f32x2{v[u].x, v[u].y};
      if (second) *(f32x2 *)(at + N) = f32x2{v[u].z, v[u].w};
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) sq[i / C] += (double)v[u][i] * (double)v[u][i];
  }
  double rms[R];
  if (norm.kind == kNormRms) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) sq[r] += __shfl_xor(sq[r], o);
      if ((threadIdx.x & 63) == 0) red[r][threadIdx.x >> 6] = sq[r];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) {
      double total = 0.0;
      for (int w = 0; w < (int)blockDim.x >> 6; ++w) total += red[r][w];
      rms[r] = sqrt(total / (double)N + norm.eps);
    }
  }
#pragma unroll
  for (int u = 0; u < kMost; ++u) {
    const int col = C * (threadIdx.x + u * blockDim.x);
    if (col >= N) continue;
    f32x4 n;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float gamma = norm.gamma ? norm.gamma[col + i % C] : 1.f;
      n[i] = norm.kind == kNormRms ? (float)(((double)v[u][i] / rms[i / C]) * (double)gamma)
                                   : __fadd_rn(__fmul_rn(tanhf(__fmul_rn(norm.alpha, v[u][i])), gamma), norm.beta[col + i % C]);
    }
    float *out = norm.rows + (long long)row * N + col;
    if constexpr (R == 1) {
      if (norm.planes)
        store_planes(norm.rows, row, g.T, col, N, n);
      else
        *(f32x4 *)out = n;
    } else {
      *(f32x2 *)out = f32x2{n.x, n.y};
      if (second) *(f32x2 *)(out + N) = f32x2{n.z, n.w};
    }
  }
}

// Any shape (K or N not a multiple of 4, unaligned rows): one thread per element of y, W read
// coalesced along n.  For the small odd shapes of tests; the MFMA kernel takes everything else.
__global__ __launch_bounds__(256) void sgemm_plain_kernel(const float *__restrict__ x, long long xs,
                                                          const float *__restrict__ w, float *__restrict__ y,
                                                          const float *__restrict__ res, int T, int K, int N,
                                                          const float *__restrict__ bias, Activation act) {
  const int n = blockIdx.x * 256 + threadIdx.x;
  if (n >= N) return;
  for (int t = blockIdx.y; t < T; t += gridDim.y) {  // the grid's second dimension ends at 65535
    const float *xr = x + (long long)t * xs;
    float acc = 0.f;
    for (int k = 0; k < K; ++k) acc += xr[k] * w[(long long)k * N + n];
    if (bias) acc = activate(act, acc + bias[n]);
    const long long o = (long long)t * N + n;
    y[o] = res ? res[o] + acc : acc;
  }
}

}  // namespace

namespace {

// workgroups the chip runs at once: two of four wavefronts per compute unit, or one of eight
int slots_of(int wn) { return wn == 4 ? 256 : 512; }

// Steps per workgroup of sgemm_stream_kernel: as many pieces as leave no compute unit without one, in whole rounds of its
// four register sets.
int stream_quota(int tiles, int steps) {
  int pieces = 256 / tiles;
  if (pieces > 16) pieces = 16;
  if (pieces < 1) pieces = 1;
  return ((steps + pieces - 1) / pieces + 3) / 4 * 4;
}

// W of one part: the tile of sgemm_stream_kernel by an estimate of its time, and whether that kernel is the one to take.
// Rounds of workgroups times steps times what a step takes, and for pieces 2.95 us and 0.416 us per MB of them written and
// read: fitted to what each of the four tiles and 128 x 256 take for 80 products of 8 to 1400 rows, K 32 to 8192, N 32 to 16384, of which
// the choice loses 0.9 % to the best of the five, and 1.9 % of 342 others of 9 to 777 rows.  (Tiles of 32 x 128 at 0.475 us a step would take 14.0 us
// where those of 32 x 64 take 15.0 for 65 to 96 rows of 2048 -> 2048, but their errors are larger: 8.05 against 7.96e-8 there, 10.4 against 9.3 for
// 17 rows of 8192 -> 1536.)  Where a workgroup has more steps than `most`, 15 to 21 us of them, or one round of workgroups does
// not do, the larger tiles, which read W less often, are level or ahead, and so they are of a loop of four steps in tiles of 96 rows (us,
// this | 128 x 256): 256 rows of 2048 -> 2048 19.0 | 23.1, 2048 -> 3072 25.6 | 25.5, 2048 -> 4608 35 | 30; 400 rows of 2048 -> 1536 21.4 |
// 23.8; 512 rows of 1024 -> 1024 12.6 | 21, 1024 -> 3072 20.8 | 25.2; 777 rows of 1024 -> 1024 16.6 | 24.3, 1024 -> 2048 22.1 | 26.0,
// 1024 -> 3072 35 | 30; 1400 rows of 2048 -> 1024 34 | 31; rounds: 512 rows of 128 -> 16384 30 | 15, 2048 rows of 128 -> 4096 31 | 17.  The
// tile that is within these bounds may be the second best, up to a quarter behind: the sums of 128 x 256 are longer, and their errors twice as large
// (us and 1e-8 of the norm, this | 128 x 256: 512 rows of 2048 -> 1024 18.2 and 8.1 | 23.4 and 14.0, 777 rows of 1536 -> 1536 28.9 and 8.0 | 25.1 and 17.3,
// 257 rows of 1280 -> 4608 28.3 and 7.7 | 26.7 and 19.0, 1700 rows of 8192 -> 64 21.9 and 9.4 | 29.0 and 25.3).
// few: rows that this kernel takes in any case.  short_rounds: its loop is of four steps, and in several rounds.
bool choose_stream(GemmPlan &p, int T, int K, int N, bool few, bool &short_rounds) {
  const struct { int mb, kg; float step; int most; } shapes[] = {{1, 2, 0.483f, 44}, {1, 4, 0.563f, 36}, {2, 2, 0.506f, 32}, {3, 2, 0.643f, 24}};
  float least = INFINITY, least_fitting = INFINITY;
  int fitting_mb = 0, fitting_kg = 0;
  p.mb = 3;
  p.kg = 2;
  for (const auto &s : shapes) {
    const long long tiles = (T + 32 * s.mb - 1) / (32 * s.mb) * (((long long)N * s.kg + 255) / 256);
    if (tiles > 1 << 20) continue;  // (many rounds: not this kernel's anyway)
    const int steps = (K + 16 * s.kg - 1) / (16 * s.kg), quota = stream_quota((int)tiles, steps), pieces = (steps + quota - 1) / quota;
    const long long wgs = tiles * pieces;
    const float turns = (float)((wgs + 255) / 256) * quota * s.step;
    const float us = turns + (pieces > 1 ? 2.95f + 0.416e-6f * 8 * 32 * s.mb * (256 / s.kg) * wgs : 0.f);
    const float fitting = turns > 17.f ? 1.05f * us : us;  // (long loops are the estimate's weak side: 512 rows of 2048 -> 1024, 32 x 64 21.7 | 64 x 128 19.7)
    if (fitting < least_fitting && wgs <= 256 && quota <= s.most && !(s.mb == 3 && quota == 4)) {
      least_fitting = fitting;
      fitting_mb = s.mb;
      fitting_kg = s.kg;
    }
    if (us >= least) continue;
    least = us;
    short_rounds = wgs > 256 && quota == 4;
    p.mb = s.mb;
    p.kg = s.kg;
  }
  const bool fits = fitting_mb > 0 && least_fitting <= 1.24f * least;  // (none: more tiles than this kernel is asked for)
  if (fits && !few) {
    p.mb = fitting_mb;
    p.kg = fitting_kg;
  }
  return fits;
}

// The tile, by what was measured (us, 2048 -> 3072 | 2048 -> 2048 | 2048 -> 16384 | 8192 -> 2048 | 1024 -> 8192):
//   rows   32 x 128 (few)              128 x 128                  128 x 256                  256 x 256
//     45   16 | 15 | 41 | 31 | 16      23 | 19 | 59 | 37 | 24
//     96   19 | 16 | 60 | 35 | 22      22 | 21 | 62 | 37 | 24
//    128   20 | 19 | 67 | 42 | 24      22 | 20 | 63 | 41 | 24
//    160   24 | 20 | 88 | 50 | 30      30 | 26 | 102 | 59 | 34
//    256   33 | 24 | 125 | 72 | 35     31 | 27 | 105 | 61 | 37    31 | 27 | 108 | 59 | 37
//    512                               47 | 37 | 185 | 106 | 57   45 | 36 | 177 | 102 | 58   52 | 44 | 192 | 100 | 64
//   1024                               87 | 58 | 360 | 197 | 96   82 | 57 | 342 | 186 | 88   80 | 63 | 315 | 173 | 116
//   2048                               148 | 100 | 717 | 372 | 187  143 | 99 | 674 | 346 | 181  144 | 100 | 619 | 323 | 164
// W of one part (us; 128 x 128 | 128 x 256 | 256 x 256), the same products:
//    256   26 25 30 | 24 24 26 | 75 65 70 | 50 43 53 | 32 35 40
//    512   35 32 41 | 30 28 38 | 120 99 112 | 77 60 69 | 43 41 49
//    777   49 45 53 | 40 35 45 | 219 184 172 | 115 95 103 | 67 61 71
//   2048   97 85 90 | 69 61 68 | 471 391 349 | 240 197 193 | 123 106 96
// so 128 x 128 is not among its tiles.  Where weights of three parts take tiles of 32 rows, those of one take
// sgemm_stream_kernel, and 256 x 256 is chosen by the same rule for both, because the sums of 128 x 256 are longer and
// their error larger (1e-7 of the norm, the three-part product | 128 x 256 | now): 150 rows of 2048 -> 16384 1.02 | 3.42 |
// 0.96 (62.5 and 60 us), 8192 -> 2048 1.09 | 2.53 | 0.98 (41, 40), 777 rows of 8192 -> 2048 3.49 | 4.94 | 3.49 (100, 107), 1400
// rows 4.41 | 7.02 | 4.41 (173, 150), of 2048 -> 3072 2.79 | 3.16 | 2.79.
// A low tile wastes least on few rows, and reads small weights again from the L2 for little: up to 96 rows always, up to
// 256 where the higher tile would be a fifth padding or the weights are small.
// The largest needs long runs: at least 36 steps a workgroup.  Less than a round of its tiles is cut into pieces for the
// second kernel (never one shared by waiting); of more than a round the last one must be empty or at least half
// full, or the waits for shared tiles cost more than the tile saves (2048 -> 8192, 128 x 256 | 256 x 256, us: 288 tiles
// of 256 x 256 433 | 503, 320 421 | 474, 352 459 | 502, 384 496 | 468, 448 576 | 548, 544 744 | 785, 576 742 | 757,
// 640 824 | 759, 704 909 | 846; 4096 -> 8192: 320 802 | 896, 384 973 | 887; 8192 -> 8192: 288 1671 | 1873).
void choose_tile(GemmPlan &p, int T, int K, int N) {
  p.wn = 2;
  const long long weights = (long long)K * N, rows1 = (T + 31) / 32 * 32LL, rows2 = (T + 127) / 128 * 128LL;
  p.few = T <= 96 || (T <= 256 && (weights <= (T <= 128 ? 12 : 5) << 20 || rows2 * 100 >= rows1 * 125));
  if (p.parts == 1) {
    const bool low = p.few;
    bool short_rounds = false;
    p.few = choose_stream(p, T, K, N, low, short_rounds) || low;
    // (its loop goes by four steps: of up to 64 long rows most are empty, and many rounds of four do not pay, either; as many
    // sums in tiles of 32 rows, us, this | three parts: 48 rows of 32 -> 32000 8.7 | 7.2, 200 rows 29 | 20, 97 rows of 64 -> 32000
    // 15.8 | 14.2, of 128 18.7 | 17.5, but of 128 -> 16384 9.4 | 10.7)
    if (low && (K <= 64 || short_rounds)) p.parts = 3;
  }
  p.few = p.few && 2LL * kFewStep * N * 4 < 0xffffffffLL;  // (32-bit offsets into a step's rows, 64 at most)
  if (p.few && p.parts == 1) return;
  p.mb = 1;
  if (p.few) return;
  p.mb = 2;
  if (T <= 256 && p.parts == 3) return;
  p.wn = 4;
  if (T <= 256) return;
  const long long rows4 = (T + 255) / 256 * 256LL;
  const long long tiles = rows4 / 256 * ((N + 255) / 256), run = tiles * p.steps / slots_of(4);
  const long long last = tiles % slots_of(4);
  const bool fills = tiles < slots_of(4) ? 2 * run < p.steps : last == 0 || 2 * last >= slots_of(4);
  if (rows4 * 100 <= rows2 * 115 && run >= 36 && fills) p.mb = 4;
}

}  // namespace

static int tile_rows(const GemmPlan &p) { return (p.few ? 32 : 64) * p.mb; }
static int tile_columns(const GemmPlan &p) { return p.few && p.parts == 1 ? 256 / p.kg : 64 * p.wn; }
static int step_k(const GemmPlan &p) { return !p.few ? p.parts == 1 ? kWideStep : TK : p.parts == 1 ? 16 * p.kg : kFewStep; }

void describe_gemm(const GemmPlan &p, int K, int plan[7]) {
  plan[0] = !p.mfma ? 0 : p.few ? 1 : 2;
  plan[1] = p.mfma ? tile_rows(p) : 1;
  plan[2] = p.mfma ? tile_columns(p) : 1;
  plan[3] = p.workgroups;
  plan[4] = p.pieces > 1 ? p.pieces : 1;
  plan[5] = p.flag_words && p.quota % p.steps != 0;
  plan[6] = p.mfma && K % step_k(p) != 0;
}

bool gemm_takes_planes(const GemmPlan &p, int K) { return p.mfma && p.parts == 1 && !p.few && K % kWideStep == 0; }

// (the norm of a row takes a workgroup of up to 1024 threads, two registers of four each)
bool gemm_takes_next(const GemmPlan &p, int T, int N, const GemmNext &next) {
  if (!p.mfma) return false;
  // (by the kernel that adds the pieces, or by the product itself, but for three-part weights in tiles of 32 rows, and of 256 x 256, whose
  // activations nothing else of a compute unit runs beside: us, a launch of its own behind it | in it, 777 rows of 2048 -> 2 x 8192 360 | 380,
  // 1024 rows 373 | 390, 2048 rows of 1024 -> 2 x 4096 194 | 207; a block of 24 shapes 1 % slower on average)
  if (next.swiglu) return !next.norm.rows && N % 8 == 0 && (p.pieces > 1 || !(p.parts == 3 && (p.few || p.mb == 4)));
  if (p.pieces <= 1 || (next.norm.planes && (p.parts != 1 || N % 32 != 0))) return false;
  if (const GemvPrep *q = next.prep)
    return !next.norm.rows && !q->q_norm && !q->k_norm && !q->b_q && !q->b_k && !q->b_v && q->rope_tab && q->hd % 8 == 0 &&
           (long long)(q->H + 2 * q->KV) * q->hd == N && q->start_pos >= 0 && q->start_pos + T <= q->cap &&
           !(((uintptr_t)q->q_rot | (uintptr_t)q->kc | (uintptr_t)q->vc) & 15);
  return N % 4 == 0 && N / (p.parts == 1 ? 4 : 2) <= 2048;
}

GemmPlan plan_gemm(int T, int K, int N, long long x_stride, bool w_bf16) {
  GemmPlan p = {};
  p.parts = w_bf16 ? 1 : 3;
  // (the kernel addresses the rows of x by 32-bit byte offsets from a base that moves along K)
  p.mfma = T >= 1 && K >= 4 && N >= 4 && (K & 3) == 0 && (N & 3) == 0 && (x_stride & 3) == 0 &&
           (long long)T * x_stride * 4 < 0xffffffffLL && (long long)TK * N * 4 < 0xffffffffLL;
  p.steps = (K + TK - 1) / TK;
  choose_tile(p, T, K, N);
  const int TN = tile_columns(p), TM = tile_rows(p);
  p.steps = (K + step_k(p) - 1) / step_k(p);
  p.tiles_m = (T + TM - 1) / TM;
  p.tiles_n = (N + TN - 1) / TN;
  if (!p.mfma) return p;
  const int slots = slots_of(p.wn);
  const int tiles = p.tiles_m * p.tiles_n;
  // groups of workgroups that stay on the same XCDs: as many (of 8, 4, 2, 1) as divide the tiles evenly
  p.group_bits = 3;
  while (tiles & ((1 << p.group_bits) - 1)) --p.group_bits;
  const int groups = 1 << p.group_bits;
  p.tiles_per_group = tiles / groups;
  if (p.few && p.parts == 1) {
    p.quota = stream_quota(tiles, p.steps);
    p.pieces = (p.steps + p.quota - 1) / p.quota;
    p.workgroups = tiles * p.pieces;
    if (p.pieces > 1) p.partial_floats = (size_t)p.workgroups * TM * TN;
    return p;
  }
  if (p.few) {  // pieces of about twelve steps, more where that leaves compute units without one, of at least four steps each
    int pieces = p.steps / 12 > 256 / tiles ? p.steps / 12 : 256 / tiles;
    if (pieces > slots / tiles) pieces = slots / tiles;
    if (pieces > 16) pieces = 16;
    if (pieces > p.steps / 4) pieces = p.steps / 4;
    if (pieces < 1) pieces = 1;
    p.quota = (p.steps + pieces - 1) / pieces;
    p.workgroups = tiles * pieces;
    p.pieces = pieces;
    if (pieces > 1) p.partial_floats = (size_t)p.workgroups * TM * TN;
    return p;
  }
  if (tiles % slots == 0) {  // whole rounds of the chip: a workgroup per tile
    p.quota = p.steps;
    p.workgroups = tiles;
    return p;
  }
  // Otherwise one round of workgroups shares the K steps of all tiles evenly.
  const long long units = (long long)p.tiles_per_group * p.steps;
  const int sixteen = step_k(p) / TK, least = 16 / sixteen;  // (16 steps of 16: a workgroup's start and end must not outweigh its loop)
  int places = slots / groups;
  int quota = (int)((units + places - 1) / places);
  if (quota < least) quota = p.steps < least ? p.steps : least;
  if (2 * quota >= p.steps) {  // a tile is shared by two or three workgroups: the one that ends it adds the pieces
    p.quota = quota;
    p.workgroups = (int)((units + quota - 1) / quota) * groups;
    p.flag_words = (size_t)p.workgroups;
  } else {
    // more pieces per tile: as many as fill one round, of at least 8 steps each, all equal; the
    // second kernel adds them
    int pieces = slots / tiles;
    static const int pieces_knob = getenv("SHAINET_HIP_GEMM_PIECES") ? atoi(getenv("SHAINET_HIP_GEMM_PIECES")) : 0;
    if (pieces > 16) pieces = 16;  // (45 rows of 8192 -> 2048: 32 pieces 35.2 us, 16 pieces 30.7 us)
    if (pieces_knob > 0) pieces = pieces_knob;  // SHAINET_HIP_GEMM_PIECES: a tuning knob
    if (pieces > p.steps * sixteen / 8) pieces = p.steps * sixteen / 8;
    if (pieces < 1) pieces = 1;
    p.quota = (p.steps + pieces - 1) / pieces;
    p.pieces = pieces;
    p.workgroups = tiles * pieces;
    if (pieces == 1) return p;  // (short K: a workgroup per tile after all)
  }
  p.partial_floats = (size_t)p.workgroups * TM * TN;
  return p;
}

namespace {

// The kernel that adds the pieces; a lane of the product holds COLUMNS neighbouring columns.  (Rows go along the grid's second dimension,
// which ends at 65535: no product of as many is cut into pieces.)
template <int COLUMNS>
hipError_t launch_sum(const GemmArgs &g, const PieceShape &s, const GemmNext &next, hipStream_t stream) {
  constexpr int R = COLUMNS == 2 ? 2 : 1, C = 4 / R;
  const int N = next.swiglu ? g.N / 2 : g.N, quads = (N + C - 1) / C, rows = (g.T + R - 1) / R;
  if (next.prep) {
    hipLaunchKernelGGL((sgemm_sum_prep_kernel<COLUMNS>), dim3((unsigned)((quads / 2 + 255) / 256), (unsigned)rows), dim3(256), 0, stream, g, s,
                       *next.prep);
    return hipGetLastError();
  }
  if (next.norm.rows) {
    const int threads = quads < 1024 ? (quads + 63) / 64 * 64 : 1024;
    hipLaunchKernelGGL((sgemm_sum_norm_kernel<COLUMNS>), dim3((unsigned)rows), dim3(threads), 0, stream, g, s, next.norm);
    return hipGetLastError();
  }
  const int threads = quads < 256 ? (quads + 63) / 64 * 64 : 256;
  const dim3 grid((unsigned)((quads + threads - 1) / threads), (unsigned)rows);
  if (next.swiglu)
    hipLaunchKernelGGL((sgemm_sum_kernel<COLUMNS, true>), grid, dim3(threads), 0, stream, g, s);
  else
    hipLaunchKernelGGL((sgemm_sum_kernel<COLUMNS, false>), grid, dim3(threads), 0, stream, g, s);
  return hipGetLastError();
}

template <int WM, int WN, int MB>
hipError_t launch_tiles(const GemmArgs &g, const GemmPlan &p, const GemmNext &next, hipStream_t stream) {
  const dim3 grid((unsigned)p.workgroups), block(64 * WM * WN);
  constexpr bool kSwiglu = MB < 4;  // (the others leave it to a launch of its own)
  const bool swiglu = next.swiglu && !g.pieces;
  if (swiglu && !kSwiglu) return hipErrorInvalidValue;
  if (swiglu && g.K % TK != 0)
    hipLaunchKernelGGL((sgemm_split_kernel<WM, WN, MB, true, kSwiglu>), grid, block, 0, stream, g);
  else if (swiglu)
    hipLaunchKernelGGL((sgemm_split_kernel<WM, WN, MB, false, kSwiglu>), grid, block, 0, stream, g);
  else if (g.K % TK != 0)
    hipLaunchKernelGGL((sgemm_split_kernel<WM, WN, MB, true, false>), grid, block, 0, stream, g);
  else
    hipLaunchKernelGGL((sgemm_split_kernel<WM, WN, MB, false, false>), grid, block, 0, stream, g);
  const hipError_t e = hipGetLastError();
  return e != hipSuccess || !g.pieces ? e : launch_sum<2>(g, PieceShape{32 * WM * MB, 64 * WN, 32 * MB, WN, 64 * WM * WN}, next, stream);
}

template <int WM, bool PLANES>
hipError_t launch_wide(const GemmArgs &g, const GemmPlan &p, const GemmNext &next, hipStream_t stream) {
  const dim3 grid((unsigned)p.workgroups);
  const bool swiglu = next.swiglu && !g.pieces;
  const int end = g.K % kWideStep == 0 ? kWhole : g.K > kWideStep ? kShifted : kGuarded;
  if (end != kWhole && PLANES) return hipErrorInvalidValue;
#define SHAINET_WIDE_LAUNCH(END_)                                                                          \
  do {                                                                                                     \
    if (swiglu)                                                                                            \
      hipLaunchKernelGGL((sgemm_wide_kernel<WM, END_, true, PLANES>), grid, dim3(512), 0, stream, g);      \
    else                                                                                                   \
      hipLaunchKernelGGL((sgemm_wide_kernel<WM, END_, false, PLANES>), grid, dim3(512), 0, stream, g);     \
  } while (0)
  if (end == kWhole)
    SHAINET_WIDE_LAUNCH(kWhole);
  else if (end == kShifted)
    SHAINET_WIDE_LAUNCH(PLANES ? kWhole : kShifted);
  else
    SHAINET_WIDE_LAUNCH(PLANES ? kWhole : kGuarded);
#undef SHAINET_WIDE_LAUNCH
  const hipError_t e = hipGetLastError();
  return e != hipSuccess || !g.pieces ? e : launch_sum<2 * WM>(g, PieceShape{64 * WM, 256, 64, 8 / WM, 512}, next, stream);
}

hipError_t launch_few(const GemmArgs &g, const GemmPlan &p, const GemmNext &next, hipStream_t stream) {
  const dim3 grid((unsigned)p.workgroups);
  if (g.K % kFewStep != 0)
    hipLaunchKernelGGL((sgemm_few_kernel<true>), grid, dim3(256), 0, stream, g);
  else
    hipLaunchKernelGGL((sgemm_few_kernel<false>), grid, dim3(256), 0, stream, g);
  const hipError_t e = hipGetLastError();
  return e != hipSuccess || !g.pieces ? e : launch_sum<2>(g, PieceShape{32, 128, 32, 2, 128}, next, stream);
}

template <int MB, int KG>
hipError_t launch_stream(const GemmArgs &g, const GemmPlan &p, const GemmNext &next, hipStream_t stream) {
  const dim3 grid((unsigned)p.workgroups);
  const bool guard = g.K % (16 * KG) != 0, swiglu = next.swiglu && !g.pieces;
  if (swiglu && guard)
    hipLaunchKernelGGL((sgemm_stream_kernel<MB, KG, true, true>), grid, dim3(512), 0, stream, g);
  else if (swiglu)
    hipLaunchKernelGGL((sgemm_stream_kernel<MB, KG, false, true>), grid, dim3(512), 0, stream, g);
  else if (guard)
    hipLaunchKernelGGL((sgemm_stream_kernel<MB, KG, true, false>), grid, dim3(512), 0, stream, g);
  else
    hipLaunchKernelGGL((sgemm_stream_kernel<MB, KG, false, false>), grid, dim3(512), 0, stream, g);
  const hipError_t e = hipGetLastError();
  return e != hipSuccess || !g.pieces ? e : launch_sum<1>(g, PieceShape{32 * MB, 256 / KG, 0, 0, 0}, next, stream);
}

}  // namespace

hipError_t launch_gemm(const float *x, long long x_stride, const float *w, float *y, const float *res, float *partials,
                       unsigned *flags, int *error, int T, int K, int N, const GemmPlan &p, hipStream_t stream,
                       unsigned *flag_set, int spin_limit, const float *bias, Activation act, const GemmNext &next, bool planes) {
  if (planes && !gemm_takes_planes(p, K)) return hipErrorInvalidValue;
  const bool more = next.swiglu || next.norm.rows || next.prep;
  if (more && !gemm_takes_next(p, T, N, next)) return hipErrorInvalidValue;
  if (!x || !w || !y || T < 1 || K < 1 || N < 1 || x_stride < K) return hipErrorInvalidValue;
  const bool aligned = !(((uintptr_t)x | (uintptr_t)w | (uintptr_t)y | (uintptr_t)res | (uintptr_t)bias | (uintptr_t)next.norm.rows) & 15);
  if (!aligned && (more || planes)) return hipErrorInvalidValue;
  if (!p.mfma || !aligned) {
    hipLaunchKernelGGL(sgemm_plain_kernel, dim3((unsigned)((N + 255) / 256), (unsigned)(T < 65535 ? T : 65535)), dim3(256), 0, stream, x,
                       x_stride, w, y, res, T, K, N, bias, act);
    return hipGetLastError();
  }
  if (p.partial_floats && !partials) return hipErrorInvalidValue;
  if (p.flag_words && (!flags || !error)) return hipErrorInvalidValue;
  GemmArgs g = {};
  g.x = planes ? nullptr : x;
  g.xs = x_stride;
  g.planes = planes ? (const unsigned short *)x : nullptr;
  g.w = w;
  g.y = y;
  g.res = res;
  g.bias = bias;
  g.act = act;
  g.partials = partials;
  g.flags = flags;
  g.flag_set = flag_set ? flag_set : flags;
  g.spin_limit = spin_limit > 0 ? spin_limit : 1 << 21;  // polls of about a microsecond each: seconds
  g.error = error;
  g.T = T;
  g.K = K;
  g.N = N;
  g.tiles_m = p.tiles_m;
  g.steps = p.steps;
  g.group_bits = p.group_bits;
  g.tiles_per_group = p.tiles_per_group;
  g.quota = p.quota;
  g.pieces = p.pieces > 1 ? p.pieces : 0;
  if (p.parts == 1) {
    if (p.few && p.kg == 4) return launch_stream<1, 4>(g, p, next, stream);
    if (p.few) return p.mb == 1 ? launch_stream<1, 2>(g, p, next, stream) : p.mb == 2 ? launch_stream<2, 2>(g, p, next, stream) : launch_stream<3, 2>(g, p, next, stream);
    if (planes) return p.mb == 4 ? launch_wide<4, true>(g, p, next, stream) : launch_wide<2, true>(g, p, next, stream);
    return p.mb == 4 ? launch_wide<4, false>(g, p, next, stream) : launch_wide<2, false>(g, p, next, stream);
  }
  if (p.few) return launch_few(g, p, next, stream);
  if (p.wn == 4) return p.mb == 4 ? launch_tiles<2, 4, 4>(g, p, next, stream) : launch_tiles<2, 4, 2>(g, p, next, stream);
  return launch_tiles<2, 2, 2>(g, p, next, stream);
}

}  // namespace shainet
