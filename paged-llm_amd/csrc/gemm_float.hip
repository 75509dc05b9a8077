// C[M, N] = A[M, K] * W[N, K]^T with float operands, float products and float sums on the matrix cores
// (v_mfma_f32_16x16x4_f32: a fused multiply-add per element, no narrower type anywhere), for any M, N, K and strides.
// This is every matrix product of the true 32-bit path.
//
// One order of additions for every shape.  K is cut into 16 slices of whole steps of 32 (the slice length depends on K
// alone); a wavefront sums its slice in ascending k, slices 2i and 2i + 1 are added, and the eight pair sums are added in
// ascending order.  How many rows a product has, and which tile or form of the kernel an element falls into, changes none
// of that: the same row gives the same bits in any batch.  (The sums are also sixteen times shorter than one running sum
// over K: relative error against 64 bits 2.1e-7 at K = 2048 and 3.4e-7 at 5632.)
//
// Why slices as wavefronts.  A wavefront holds a tile of (16 MT) rows x (16 NT) weight rows and loads both operands
// straight into the matrix instruction's registers (16 bytes a lane; lane l holds row l % 16, columns 4 (l / 16) .. + 3 of
// sixteen columns, and element j of every lane makes the j-th of four instructions).  The slices need nothing from each
// other until they are added through LDS at the end, so there is no barrier in the loop.
//   * Few rows (decoding): bound by the weights' way from memory.  Sixteen wavefronts, one slice each, in tiles of 16 x 16
//     or 16 x 32 (2048 weight rows are 128 workgroups) and at most 64 registers, so that two workgroups share a compute
//     unit: 8 rows x 2048 x 2048 in 9.0 us, 11264 x 2048 in 24.9 us (3.7 TB/s), 2048 x 5632 in 20.8 us, where a kernel of 64 x 64
//     outputs with all of K in one workgroup took 288, 287 and 798 us.  More loads under way (four steps of 32 instead of
//     two) changed nothing at two workgroups less per compute unit.
//   * Many rows: bound by the matrix cores (157 TFLOP/s at the nominal clock) while a tile of 64 x 64 draws 16 bytes a clock
//     and compute unit from the L2.  Eight wavefronts take two slices each, one after the other, with 216 registers a
//     lane: 2048 rows x 2048 x 5632 in 445 us (106 TFLOP/s), 301 rows x 2048 x 5632 in 86 us (tiles of 48 x 64 fill the GPU in
//     one round; 1027 us before).
//   * Short K (the matrices of heads): bound by memory and by what a workgroup takes to start and end.  Only the wavefronts that
//     have columns are launched, one for every slice or two of 32 (64 heads of 64 x 64 at 300 / 1500 rows: 6.9 / 20 us, 2.5 TB/s at
//     the latter; the kernel with all of K in one workgroup's LDS tiles took 13.5 / 29).
// Rows that 16-byte loads cannot take (K or a stride no multiple of 4) are read element by element in the same places: 8 / 301 /
// 1024 rows x 2048 x 2047 in 11.9 / 41 / 98 us.
// Which tile a product takes is the host's choice by the rounds of workgroups (ops.float_gemm_plan).
#include "common.h"

using namespace pllm;

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kSlices = 16, kSliceUnit = 32;

struct FloatGemm {
  const float* A;
  const float* W;
  float* C;
  long a_batch, w_batch, c_batch;
  int lda, ldw, ldc, M, N, K, slice, row_tiles, col_tiles;
};

// Four consecutive elements of a row from column k on; zeros from column K on.  VEC: K and the row's start are multiples
// of four elements, so the four lie on either side of K together.
template <bool VEC>
__device__ __forceinline__ f32x4 load_quad_tail(const float* row, int k, int K) {
  if (VEC) return k < K ? *reinterpret_cast<const f32x4*>(row + k) : f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 v;
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = k + j < K ? row[k + j] : 0.f;
  return v;
}
template <bool VEC>
__device__ __forceinline__ f32x4 load_quad(const float* p) {
  if (VEC) return *reinterpret_cast<const f32x4*>(p);
  return f32x4{p[0], p[1], p[2], p[3]};
}

// ALL: every slice has columns, and the workgroup all its wavefronts.
template <int MT, int NT, int SPW, int HALVES, int DEPTH, int PER_SIMD, bool VEC, bool ALL>
__global__ __launch_bounds__(64 * (kSlices / SPW), PER_SIMD) void gemm_float_kernel(FloatGemm g) {
  constexpr int kStep = 16 * HALVES;
  extern __shared__ __attribute__((aligned(16))) unsigned char gf_lds[];
  f32x4* parts = reinterpret_cast<f32x4*>(gf_lds);                     // [wavefronts][MT * NT][64]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, quad = lane >> 4;

  // The row tiles of one tile of weight rows follow each other on one XCD (workgroup b runs on XCD b % 8), so that its L2
  // hands the weights from one to the next.  The last group has fewer than eight tiles of weight rows where their number is no
  // multiple of 8: its workgroups go round the XCDs all the same (64 heads of 64 x 64 at 1500 rows: 20 us; 278 with the
  // group filled up by workgroups without work, which left the others on one XCD, and with sixteen wavefronts for two slices).
  const int b = blockIdx.x, group = b / (g.row_tiles * 8), in_group = b - group * g.row_tiles * 8, across = min(8, g.col_tiles - group * 8);
  const int row_tile = across == 8 ? in_group >> 3 : in_group / across, col_tile = group * 8 + in_group - row_tile * across;
  const int m0 = row_tile * (16 * MT), n0 = col_tile * (16 * NT);
  const float* A = g.A + (size_t)blockIdx.y * g.a_batch;
  const float* W = g.W + (size_t)blockIdx.y * g.w_batch;
  float* C = g.C + (size_t)blockIdx.y * g.c_batch;

  const float *a_row[MT], *w_row[NT];                                  // rows past the end repeat the last one
#pragma unroll
  for (int i = 0; i < MT; ++i) a_row[i] = A + (size_t)min(m0 + 16 * i + r16, g.M - 1) * g.lda + 4 * quad;
#pragma unroll
  for (int i = 0; i < NT; ++i) w_row[i] = W + (size_t)min(n0 + 16 * i + r16, g.N - 1) * g.ldw + 4 * quad;

  f32x4 total[MT * NT];
#pragma unroll
  for (int s = 0; s < SPW; ++s) {
    const int begin = min((wave * SPW + s) * g.slice, g.K), end = min(begin + g.slice, g.K);
    const int steps = (end - begin) / kStep;                           // whole steps; the last slice may have a tail
    f32x4 acc[MT * NT];
#pragma unroll
    for (int i = 0; i < MT * NT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](const f32x4* a, const f32x4* w) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int n = 0; n < NT; ++n) acc[i * NT + n] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[n][j], a[i][j], acc[i * NT + n], 0, 0, 0);
    };
    if (steps > 0) {
      f32x4 a[DEPTH][HALVES][MT], w[DEPTH][HALVES][NT];
      auto fetch = [&](int stage, int step) {
        const int k = begin + step * kStep;
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
          for (int h = 0; h < HALVES; ++h) w[stage][h][n] = load_quad<VEC>(w_row[n] + k + 16 * h);
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int h = 0; h < HALVES; ++h) a[stage][h][i] = load_quad<VEC>(a_row[i] + k + 16 * h);
      };
      auto work = [&](int stage) {
#pragma unroll
        for (int h = 0; h < HALVES; ++h) multiply(a[stage][h], w[stage][h]);
      };
#pragma unroll
      for (int d = 0; d < DEPTH; ++d) fetch(d, min(d, steps - 1));
      int at = 0;
      for (; at + 2 * DEPTH <= steps; at += DEPTH) {                   // (no condition on a load here: the waits stay exact)
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
          work(d);
          fetch(d, at + d + DEPTH);
        }
      }
#pragma unroll
      for (int d = 0; d < DEPTH; ++d) {                                // the last 1 to 2 DEPTH - 1 steps
        if (at + d >= steps) break;
        work(d);
        if (at + d + DEPTH < steps) fetch(d, at + d + DEPTH);
      }
#pragma unroll
      for (int d = 0; d < DEPTH - 1; ++d)
        if (at + d + DEPTH < steps) work(d);
    }
    for (int k = begin + steps * kStep; k < end; k += 16) {             // less than a step is left: zeros stand past the last column
      f32x4 a[MT], w[NT];
#pragma unroll
      for (int n = 0; n < NT; ++n) w[n] = load_quad_tail<VEC>(w_row[n] - 4 * quad, k + 4 * quad, g.K);
#pragma unroll
      for (int i = 0; i < MT; ++i) a[i] = load_quad_tail<VEC>(a_row[i] - 4 * quad, k + 4 * quad, g.K);
      multiply(a, w);
    }
#pragma unroll
    for (int i = 0; i < MT * NT; ++i) total[i] = s == 0 ? acc[i] : total[i] + acc[i];
  }

#pragma unroll
  for (int i = 0; i < MT * NT; ++i) parts[(wave * MT * NT + i) * 64 + lane] = total[i];
  __syncthreads();
  const bool wide = (g.ldc & 3) == 0 && (reinterpret_cast<uintptr_t>(C) & 15) == 0;
  const int threads = ALL ? 64 * (kSlices / SPW) : (int)blockDim.x;
  for (int at = tid; at < MT * NT * 64; at += threads) {
    f32x4 sum;
#pragma unroll
    for (int p = 0; p < kSlices / 2; ++p) {
      constexpr int kEach = MT * NT * 64;
      if (!ALL && p > 0 && 2 * p * g.slice >= g.K) break;              // (slices past K are zeros that change no sum: nobody makes them)
      f32x4 pair = parts[(SPW == 2 ? p : 2 * p) * kEach + at];
      if (SPW == 1 && (ALL || (2 * p + 1) * g.slice < g.K)) pair += parts[(2 * p + 1) * kEach + at];
      sum = p == 0 ? pair : sum + pair;
    }
    const int tile = at >> 6, m = m0 + 16 * (tile / NT) + (at & 15), n = n0 + 16 * (tile % NT) + 4 * ((at & 63) >> 4);
    if (m >= g.M || n >= g.N) continue;
    float* c = C + (size_t)m * g.ldc + n;
    if (wide && n + 4 <= g.N) {
      *reinterpret_cast<f32x4*>(c) = sum;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (n + j < g.N) c[j] = sum[j];
    }
  }
}

template <int MT, int NT, int SPW, int HALVES, int DEPTH, int PER_SIMD>
static int launch_float_gemm(const FloatGemm& g, int batch, bool vec, hipStream_t stream) {
  FloatGemm p = g;
  p.row_tiles = (g.M + 16 * MT - 1) / (16 * MT);
  p.col_tiles = (g.N + 16 * NT - 1) / (16 * NT);
  const int used = (g.K + g.slice - 1) / g.slice, waves = (used + SPW - 1) / SPW;     // wavefronts that have columns: 1 to kSlices / SPW
  const size_t lds = (size_t)waves * MT * NT * 64 * sizeof(f32x4);
  auto kernel = used == kSlices ? (vec ? gemm_float_kernel<MT, NT, SPW, HALVES, DEPTH, PER_SIMD, true, true> : gemm_float_kernel<MT, NT, SPW, HALVES, DEPTH, PER_SIMD, false, true>)
                                : (vec ? gemm_float_kernel<MT, NT, SPW, HALVES, DEPTH, PER_SIMD, true, false> : gemm_float_kernel<MT, NT, SPW, HALVES, DEPTH, PER_SIMD, false, false>);
  if (lds > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return (int)e;
  }
  const dim3 grid((unsigned)(p.col_tiles * p.row_tiles), batch), block(64 * waves);
  hipLaunchKernelGGL(kernel, grid, block, lds, stream, p);
  PLLM_RETURN_LAST_ERROR();
}

// `batch` products at once, operand b at its base plus b times its batch stride (elements).  `rows_tile`, `cols_tile`: the
// tile in sixteens of rows and weight rows, one of the forms below.
PLLM_API int pllm_gemm_float(const float* A, int lda, long a_batch, const float* W, int ldw, long w_batch, float* C, int ldc, long c_batch,
                             int M, int N, int K, int batch, int rows_tile, int cols_tile, hipStream_t stream) {
  if (M <= 0 || N <= 0 || batch <= 0) return 0;
  if (K <= 0 || batch > 65535) return -2;
  const int slice = (K + kSlices * kSliceUnit - 1) / (kSlices * kSliceUnit) * kSliceUnit;
  const FloatGemm g{A, W, C, a_batch, w_batch, c_batch, lda, ldw, ldc, M, N, K, slice, 0, 0};
  auto fours = [](const void* p, long a, long b) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0 && a % 4 == 0 && b % 4 == 0; };
  const bool vec = K % 4 == 0 && fours(A, lda, a_batch) && fours(W, ldw, w_batch);
  switch (rows_tile * 10 + cols_tile) {
    case 11: return launch_float_gemm<1, 1, 1, 2, 2, 8>(g, batch, vec, stream);
    case 12: return launch_float_gemm<1, 2, 1, 2, 1, 8>(g, batch, vec, stream);
    case 22: return launch_float_gemm<2, 2, 1, 2, 1, 4>(g, batch, vec, stream);
    case 34: return launch_float_gemm<3, 4, 2, 1, 2, 2>(g, batch, vec, stream);
    case 44: return launch_float_gemm<4, 4, 2, 1, 2, 2>(g, batch, vec, stream);
    default: return -3;
  }
}
