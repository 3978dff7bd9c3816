// fp32 products on the bf16 matrix cores.  A float is the exact sum of three bf16 numbers, its value
// rounded to bf16, the rest rounded to bf16, and the rest of that (8 + 8 + 8 mantissa bits with signs of
// their own).  A bf16 has a float's exponents and 16 bits less behind them, so the rests of a float below 2^-110
// would not be whole; operands are lifted by 2^24 first, which makes every part of every float, the smallest
// subnormal's too, a normal bf16 or zero, and results are brought down again.  (Not the operands of scores, see
// QueryRange, nor probabilities, whose row holds one near 1, nor the values of prefill attention, which looks at its
// sums instead.)  That is 2 to 4 % of a prompt's products; rows of x around 2^-120 had an error of 3.5e-5 without, and
// 2e-7 with it, as rows around 1 have.  Of the nine products of two such sums
// the six largest make up the product to 2^-24 of itself: of the three left out two can reach 2^-25 each.  Six
// v_mfma_f32_32x32x16_bf16 of 32 cycles do what eight v_mfma_f32_32x32x2_f32 of 64 do (192 against 512
// cycles per 32 x 32 x 16; a loop of nothing else: 1876 TFLOP/s of bf16 = 312 of fp32, against 155), they
// leave the vector ALU free meanwhile, which the fp32 instruction does not, and round the accumulator
// 6/16 times per term instead of 1/2: measured against 64 bits the error is 0.4 to 0.95 of the fp32
// instruction's for sums of 64 to 8192 terms.
// What is not finite in an operand (or infinite once it is lifted: from 2^104 on, and sums of products from 2^80
// on) makes NaN or infinity of the sums it enters; callers look for sums that are not finite and take those again
// with the fp32 instruction, its operands straight from memory: the wavefronts that meet such a value cost two to
// four times what they do otherwise.
#pragma once
#include <hip/hip_runtime.h>

#include <stdint.h>

namespace shainet {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Operands of a product are lifted before they are split; its result, or that of one lifted operand, comes down.
constexpr float kLift = 0x1p24f, kDrop = 0x1p-48f, kDropOne = 0x1p-24f;

// Scores of attention are taken of queries and keys as they are: only their size against 1 counts, and what the
// small ones lose is 2^-134 of the other operand at most.  It can count where a query (scaled, in log2 units) holds
// numbers of 2^100 and more, and keys numbers below 2^-110, or the query numbers below 2^-109 (other than 0), and keys
// very large ones: the scores of such queries are taken in fp32.
struct QueryRange {
  unsigned least = ~0u, most = 0u;  // of the bits of |q|, doubled; zeros lie above all in `least`
  __device__ __forceinline__ void add(f32x4 q) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const unsigned bits = __builtin_bit_cast(unsigned, q[i]) << 1;
      least = min(least, bits - 1u);
      most = max(most, bits);
    }
  }
  // c: what the queries are multiplied by for the scores (the multiplication itself stays with the subtractions of the
  // split, where it is not rounded)
  __device__ __forceinline__ bool apart(float c) const {
    const float lo = __builtin_bit_cast(float, (least + 1u) >> 1), hi = __builtin_bit_cast(float, most >> 1);
    return (least != ~0u && !(fabsf(lo * c) >= 0x1p-109f)) || !(fabsf(hi * c) < 0x1p100f);
  }
};

// two floats rounded to bf16, the first in the low half
__device__ __forceinline__ unsigned pack_bf16(float a, float b) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{a, b}), bf16x2));
}

// two floats that are bf16 numbers, packed the same way
__device__ __forceinline__ unsigned pack_high(float a, float b) {
  return __builtin_amdgcn_perm(__builtin_bit_cast(unsigned, b), __builtin_bit_cast(unsigned, a), 0x07060302u);
}

// the three parts of two floats, packed
__device__ __forceinline__ void split_pair(float a, float b, unsigned &high, unsigned &mid, unsigned &low) {
  high = pack_bf16(a, b);
  a -= __builtin_bit_cast(float, high << 16);
  b -= __builtin_bit_cast(float, high & 0xffff0000u);
  mid = pack_bf16(a, b);
  a -= __builtin_bit_cast(float, mid << 16);
  b -= __builtin_bit_cast(float, mid & 0xffff0000u);
  low = pack_bf16(a, b);
}

// the three parts of four floats
__device__ __forceinline__ void split_quad(f32x4 v, u32x2 &high, u32x2 &mid, u32x2 &low) {
  unsigned a[2], b[2], c[2];
  split_pair(v.x, v.y, a[0], b[0], c[0]);
  split_pair(v.z, v.w, a[1], b[1], c[1]);
  high = u32x2{a[0], a[1]};
  mid = u32x2{b[0], b[1]};
  low = u32x2{c[0], c[1]};
}

// the three parts of eight floats: a fragment of each
__device__ __forceinline__ void split_octet(f32x4 a, f32x4 b, u32x4 &high, u32x4 &mid, u32x4 &low) {
  u32x2 h[2], m[2], l[2];
  split_quad(a, h[0], m[0], l[0]);
  split_quad(b, h[1], m[1], l[1]);
  high = u32x4{h[0].x, h[0].y, h[1].x, h[1].y};
  mid = u32x4{m[0].x, m[0].y, m[1].x, m[1].y};
  low = u32x4{l[0].x, l[0].y, l[1].x, l[1].y};
}

// The parts of four lifted floats as a product takes them from memory, in three planes.  What a bf16 cannot hold lifted (not finite, or from
// 2^104 on) is NaN in the first plane, so that its sums are taken again, and stands as it is in the two others.
__device__ __forceinline__ void split_planes(f32x4 v, u32x2 (&part)[3]) {
  split_quad(v * kLift, part[0], part[1], part[2]);
  const unsigned any = 0x7f807f80u;  // exponents of all ones
  const unsigned a = part[0].x & any, b = part[0].y & any;
  if ((a & 0xffffu) == 0x7f80u || (a >> 16) == 0x7f80u || (b & 0xffffu) == 0x7f80u || (b >> 16) == 0x7f80u) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int at = 16 * (i & 1);
      const unsigned bits = __builtin_bit_cast(unsigned, (float)v[i]);
      if ((part[0][i >> 1] >> at & 0x7f80u) != 0x7f80u) continue;
      part[0][i >> 1] = (part[0][i >> 1] & ~(0xffffu << at)) | 0x7fc0u << at;
      part[1][i >> 1] = (part[1][i >> 1] & ~(0xffffu << at)) | (bits >> 16) << at;
      part[2][i >> 1] = (part[2][i >> 1] & ~(0xffffu << at)) | (bits & 0xffffu) << at;
    }
  }
}
// ... and into planes [3][cols / 32][rows][32]: four neighbouring columns of a row (of 64 bytes in a plane, so that what a product copies
// for a step of 32 along K lies together: rows of whole planes, K apart by a power of two, took 2048 rows of 8192 -> 2048 from 160 to 248 us)
__device__ __forceinline__ void store_planes(void *planes, int row, int rows, int col, int cols, f32x4 v) {
  u32x2 part[3];
  split_planes(v, part);
  unsigned short *at = (unsigned short *)planes + ((long long)(col / 32) * rows + row) * 32 + col % 32;
#pragma unroll
  for (int p = 0; p < 3; ++p) *(u32x2 *)(at + p * (long long)rows * cols) = part[p];
}
// four neighbouring floats, whole again; plane: numbers from a part to the next
__device__ __forceinline__ f32x4 join_planes(const unsigned short *at, long long plane) {
  const u32x2 h = *(const u32x2 *)at, m = *(const u32x2 *)(at + plane), l = *(const u32x2 *)(at + 2 * plane);
  f32x4 v;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    auto part = [&](const u32x2 &p) { return (i & 1 ? p[i >> 1] >> 16 : p[i >> 1] & 0xffffu) << 16; };
    const unsigned a = part(h), b = part(m), c = part(l);
    v[i] = (a & 0x7f800000u) == 0x7f800000u
               ? __builtin_bit_cast(float, b | c >> 16)
               : ((__builtin_bit_cast(float, a) + __builtin_bit_cast(float, b)) + __builtin_bit_cast(float, c)) * kDropOne;
  }
  return v;
}

// The parts of the two factors in the six products that are taken, smallest first.
constexpr int kPartA[6] = {2, 1, 0, 1, 0, 0}, kPartB[6] = {0, 1, 2, 0, 1, 0};

// acc += a b; operands as 16-byte fragments: lane l holds k = 8 (l / 32) .. + 7 of row (column) l % 32.
// D[m = 8 (r / 4) + 4 (l / 32) + r % 4][n = l % 32] in register r.
__device__ __forceinline__ f32x16 mfma_bf16(u32x4 a, u32x4 b, f32x16 acc) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
}

// The same of 16 x 16 over 32 k: lane l holds k = 8 (l / 16) .. + 7 of row (column) l % 16.
// D[m = 4 (l / 16) + r][n = l % 16] in register r.
__device__ __forceinline__ f32x4 mfma_bf16_16(u32x4 a, u32x4 b, f32x4 acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
}

// The same in fp32 over two k: lane l holds k = l / 32 of row (column) l % 32; the same D.
__device__ __forceinline__ f32x16 mfma_f32(float a, float b, f32x16 acc) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc, 0, 0, 0);
}
// ... and of 16 x 16 over four k: lane l holds k = l / 16 of row (column) l % 16; D as of mfma_bf16_16
__device__ __forceinline__ f32x4 mfma_f32_16(float a, float b, f32x4 acc) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc, 0, 0, 0); }

// *base (the same in all lanes) plus a lane's own offset in bytes: one load with a scalar base.  (Of addresses that differ
// by scalars only the compiler makes 64-bit sums per thread, two instructions each.)
template <typename V>
__device__ __forceinline__ V load_at(const V *base, unsigned offset) {
  uint64_t at = (uint64_t)base;
  asm("" : "+s"(at), "+v"(offset));
  return *(const __attribute__((address_space(1))) V *)(at + offset);
}

// The same with an offset that keeps its register over a loop.
template <typename V>
__device__ __forceinline__ V load_from(const V *base, unsigned &offset) {
  uint64_t at = (uint64_t)base;
  asm("" : "+s"(at), "+v"(offset));
  return *(const __attribute__((address_space(1))) V *)(at + offset);
}

}  // namespace shainet
