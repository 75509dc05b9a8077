// Float products on the bfloat16 matrix cores, for the kernels of the 32-bit path.
//
// A float is the sum of three bfloat16 numbers, each the rest rounded to nearest: 8 + 8 + 8 bits and their signs hold all
// 24.  Of the nine products of parts the six that reach 2^-24 of the whole are formed (exactly: 8 x 8 bits) and added in
// float by v_mfma_f32_16x16x32_bf16, the small ones first: six instructions for 32 columns where the float instruction
// takes eight of twice the time.  A chain of 32 columns is rounded six times instead of 32, so the sums are nearer to 64 bits than
// those of float products were: relative error 1.7e-7 (2.1e-7) at K = 2048, 2.9e-7 (3.4e-7) at 5632, 4.7e-8 (1.1e-7) at 64.
//
// One order of additions for every shape and kernel.  K is cut into 16 slices of whole steps of 32 columns, by K alone; a slice is one
// chain in ascending k, and the slices are added as a balanced tree, neighbours first.
//
// Infinities, NaN, and numbers that round past the largest bfloat16 have parts that cancel or meet zeros where the numbers
// themselves do not: a result that is not finite is made again by `plain_product`.
#pragma once
#include "common.h"

namespace pllm {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kSlices = 16, kStep = 32;

__host__ __device__ __forceinline__ int slice_columns(int K) { return (K + kSlices * kStep - 1) / (kSlices * kStep) * kStep; }

// A lane's eight elements of a row's 32 columns: columns 4 quad .. + 3 of both halves.
struct Octet { f32x4 lo, hi; };

struct Triple { bf16x8 part[3]; };

// (A dot product with (-1, 0) would give the rest x - part in one instruction instead of two, but it keeps the matrix cores from
// working beside it: 24 products and a split 195 ns with subtractions, 233 with dot products, 165 without a split.)
__device__ __forceinline__ Triple split(const Octet& x) {
  u32x4 part[3];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f32x2 rest = i < 2 ? f32x2{x.lo[2 * i], x.lo[2 * i + 1]} : f32x2{x.hi[2 * i - 4], x.hi[2 * i - 3]};
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      part[p][i] = __builtin_bit_cast(unsigned, __builtin_convertvector(rest, bf16x2));
      if (p < 2) rest = f32x2{rest[0] - __uint_as_float(part[p][i] << 16), rest[1] - __uint_as_float(part[p][i] & 0xffff0000u)};
    }
  }
  return {{__builtin_bit_cast(bf16x8, part[0]), __builtin_bit_cast(bf16x8, part[1]), __builtin_bit_cast(bf16x8, part[2])}};
}

// The six products, as (part of W, part of A).
constexpr int kProducts[6][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};

__device__ __forceinline__ bool finite(float x) { return fabsf(x) < INFINITY; }

// a . w over K columns from float products in ascending k, slice by slice in the same tree.
__device__ __forceinline__ float plain_product(const float* a, const float* w, int K) {
  const int slice = slice_columns(K);
  float level[5] = {0.f, 0.f, 0.f, 0.f, 0.f};                          // partial sums of the tree, one a level
#pragma unroll 1
  for (int s = 0; s < kSlices; ++s) {
    float x = 0.f;
#pragma unroll 4
    for (int k = s * slice; k < min((s + 1) * slice, K); ++k) x = fmaf(a[k], w[k], x);
#pragma unroll
    for (int l = 0, n = s; l < 4; ++l, n >>= 1) {
      if (!(n & 1)) { level[l] = x; break; }
      x = level[l] + x;
    }
    level[4] = x;
  }
  return level[4];
}

}  // namespace pllm
