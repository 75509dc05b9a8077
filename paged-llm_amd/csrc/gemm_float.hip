// C[M, N] = A[M, K] * W[N, K]^T with float operands, each the sum of three bfloat16 numbers, on the bfloat16 matrix cores
// (float_split.h: the products, the order of additions, and what is as exact as before), for any M, N, K and strides.  These are the
// matrix products of the true 32-bit path.  How many rows a product has, and which tile or form of the kernel an element
// falls into, changes no bit of it.
//
// Why slices as wavefronts.  A wavefront holds a tile of (16 MT) rows x (16 NT) weight rows of one or two slices of K.  The slices
// need nothing from each other until they are added through LDS at the end, so there is no barrier in the loop.
//   * What bounds it is the compute unit's way to the L2: four lanes that follow each other and lie in one piece of 64 bytes are taken
//     at once, lanes of different rows one by one (16 bytes a clock; the operand order of the matrix instruction has its rows in
//     neighbouring lanes).  So a load takes 8 rows x 128 bytes, and a wavefront's own corner of LDS turns them into operand order
//     (301 rows x 2048 x 2048: 25 us, 34 with loads in operand order, the same in every other arrangement tried with them).
//   * Few rows (decoding): bound by the weights' way from memory.  Sixteen wavefronts, one slice each, in tiles of 16 x 16 or 16 x
//     32 (2048 weight rows are 128 workgroups) and few enough registers for two workgroups on a compute unit: 8 rows x 2048 x 2048 in 7.2
//     us (8.8 with the float instruction, which takes the weights' loads in operand order as well), 11264 x 2048 in 22.1 (24.0), 2048 x
//     5632 in 17.1 (20.2); 64 rows x 2048 x 2048 in 10.3 (14.1).
//   * Many rows: bound by the same way (a tile of 64 x 64 draws 42 bytes a clock at the matrix cores' rate, of 45 that the L2 gives) and
//     by a wavefront's chain of load, turn, split and product.  Eight wavefronts take two slices each, one after the other, with up to 256
//     registers a lane; the first slice's sums wait in LDS.  301 rows x 2048 x 2048 / 5632 in 25 / 60 us (37 / 86 with the float
//     instruction), x 11264 x 2048 in 114 (168), 1024 rows x 2048 x 5632 in 147 (225).
//   * Short K (the matrices of heads): bound by memory and by what a workgroup takes to start and end.  Only the wavefronts that
//     have columns are launched (300 rows of 64 heads of 64 x 64: 6.2 us).
// Rows that 16-byte loads cannot take (K or a stride no multiple of 4) are read element by element in operand order.
// Which tile a product takes is the host's choice by the rounds of workgroups (ops.float_gemm_plan).
#include "float_split.h"

using namespace pllm;

struct FloatGemm {
  const float* A;
  const float* W;
  float* C;
  long a_batch, w_batch, c_batch;
  int lda, ldw, ldc, M, N, K, slice, row_tiles, col_tiles;             // N: weight rows
  // Behind the product:
  int activation, num_heads, num_kv_heads, head_dim, block_size;
  const int *positions, *slots;
  const float *cos_table, *sin_table;
  float *k_pages, *v_pages;
};

// What stands behind the product.  FG_GATED: W = [gate rows; up rows], C = act(gate) * up.  FG_ROPE_KV: W = [q; k; v] rows of heads; q and
// k are rotated, element e with e + half a head, q goes to C, k and v into the cache's pages.  Both take two weight rows for a
// result, so a tile of 16 has eight of the one kind and their eight partners.
enum { FG_PLAIN = 0, FG_GATED = 1, FG_ROPE_KV = 2 };

// The weight row that stands at place `at` (tile after tile).
template <int EPI>
__device__ __forceinline__ int weight_row(const FloatGemm& g, int at) {
  if (EPI == FG_PLAIN) return min(at, g.N - 1);                        // rows past the end repeat the last one
  const int one = (at >> 4) * 8 + (at & 7), half = EPI == FG_GATED ? g.N / 2 : g.head_dim / 2;
  if (EPI == FG_GATED) return min(one, half - 1) + ((at & 8) ? half : 0);
  const int head = one / half;
  return min(head * g.head_dim + one - head * half, g.N - half - 1) + ((at & 8) ? half : 0);
}

// ALL: every slice has columns, and the workgroup all its wavefronts.  SPW: slices of a wavefront.
template <int MT, int NT, int SPW, int PER_SIMD, int EPI, bool VEC, bool ALL>
__global__ __launch_bounds__(64 * (kSlices / SPW), PER_SIMD) void gemm_float_kernel(FloatGemm g) {
  constexpr int kPad = 272;                                            // bytes: a chunk of 16 bytes of 16 rows, and 16 against bank conflicts
  extern __shared__ __attribute__((aligned(16))) unsigned char gf_lds[];
  f32x4* parts = reinterpret_cast<f32x4*>(gf_lds + (SPW == 2 ? kSlices / SPW * 8 * kPad : 0));   // at the end: [wavefronts][MT * NT][64]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, quad = lane >> 4;
  unsigned char* turn = gf_lds + wave * 8 * kPad;                      // [8 chunks][16 rows] of 16 bytes: a tile on its way to operand order

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

  // A tile of 16 rows x 32 columns under way: two loads of 8 rows x 128 bytes, or a lane's own eight elements.
  struct Tile { f32x4 x[2]; };
  constexpr int kAt = VEC ? 2 : 1;
  const int w_first = EPI == FG_PLAIN ? n0 : 0;
  unsigned a_at[MT][kAt], w_at[NT][kAt];                               // in elements from the tile's first row; rows past the end repeat the last one
#pragma unroll
  for (int j = 0; j < kAt; ++j) {
    const int r = VEC ? 8 * j + (lane >> 3) : r16, c = VEC ? 4 * (lane & 7) : 4 * quad;
#pragma unroll
    for (int i = 0; i < MT; ++i) a_at[i][j] = (unsigned)min(16 * i + r, g.M - 1 - m0) * g.lda + c;
#pragma unroll
    for (int i = 0; i < NT; ++i) w_at[i][j] = (unsigned)(weight_row<EPI>(g, n0 + 16 * i + r) - w_first) * g.ldw + c;
  }
  const float *a_rows = A + (size_t)m0 * g.lda, *w_rows = W + (size_t)w_first * g.ldw;
  // TAIL: zeros from column K on.  (VEC: K and the row's start are multiples of four elements, so that four lie on either side of K.)
  auto load = [&](const float* rows, const unsigned* at, int k, bool tail) {
    Tile t;
    if (VEC) {
#pragma unroll
      for (int j = 0; j < kAt; ++j) t.x[j] = !tail || k + 4 * (lane & 7) < g.K ? *reinterpret_cast<const f32x4*>(rows + k + at[j]) : f32x4{0.f, 0.f, 0.f, 0.f};
    } else {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) t.x[j][e] = !tail || k + 4 * quad + 16 * j + e < g.K ? rows[(size_t)k + at[0] + 16 * j + e] : 0.f;
    }
    return t;
  };
  auto operand = [&](const Tile& t) {
    if (!VEC) return Octet{t.x[0], t.x[1]};
#pragma unroll
    for (int j = 0; j < 2; ++j) *reinterpret_cast<f32x4*>(turn + (lane & 7) * kPad + (8 * j + (lane >> 3)) * 16) = t.x[j];
    return Octet{*reinterpret_cast<f32x4*>(turn + quad * kPad + r16 * 16), *reinterpret_cast<f32x4*>(turn + (quad + 4) * kPad + r16 * 16)};
  };

  f32x4 acc[MT * NT];
  f32x4* own_part = parts + wave * MT * NT * 64 + lane;                // (SPW = 2: it holds the first slice's sums meanwhile)
  auto multiply = [&](const Triple* w, const Triple& a, int i) {
#pragma unroll
    for (int p = 0; p < 6; ++p)
#pragma unroll
      for (int n = 0; n < NT; ++n)
        acc[i * NT + n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[n].part[kProducts[p][0]], a.part[kProducts[p][1]], acc[i * NT + n], 0, 0, 0);
  };

  const int begin = min(wave * SPW * g.slice, g.K), end = min(begin + SPW * g.slice, g.K);
  const int steps = (end - begin) / kStep, per_slice = g.slice / kStep;  // whole steps; the last slice may have a tail
#pragma unroll
  for (int i = 0; i < MT * NT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (steps > 0) {
    Tile a[MT], w[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) w[n] = load(w_rows, w_at[n], begin, false);
#pragma unroll
    for (int i = 0; i < MT; ++i) a[i] = load(a_rows, a_at[i], begin, false);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll 1
    for (int step = 0; step < steps; ++step) {
      const int k = begin + min(step + 1, steps - 1) * kStep;          // (past the last step: that one again, not used)
      Triple wt[NT];
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        wt[n] = split(operand(w[n]));
        w[n] = load(w_rows, w_at[n], k, false);
      }
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const Triple at = split(operand(a[i]));
        a[i] = load(a_rows, a_at[i], k, false);
        __builtin_amdgcn_sched_barrier(0);                             // (a load that a loop hands on would be moved to its use in the next round)
        multiply(wt, at, i);
      }
      if (SPW == 2 && step + 1 == per_slice) {                         // the second slice starts from zero
#pragma unroll
        for (int i = 0; i < MT * NT; ++i) {
          own_part[i * 64] = acc[i];
          acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
      }
    }
  }
  if (begin + steps * kStep < end) {                                   // less than a step is left
    const int k = begin + steps * kStep;
    Triple wt[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) wt[n] = split(operand(load(w_rows, w_at[n], k, true)));
#pragma unroll
    for (int i = 0; i < MT; ++i) multiply(wt, split(operand(load(a_rows, a_at[i], k, true))), i);
  }
  if (SPW == 1) __syncthreads();                                       // (the sums take the place of the tiles on their way)
#pragma unroll
  for (int i = 0; i < MT * NT; ++i) own_part[i * 64] = SPW == 2 && steps >= per_slice ? own_part[i * 64] + acc[i] : acc[i];
  __syncthreads();

  const bool wide = (g.ldc & 3) == 0 && (reinterpret_cast<uintptr_t>(C) & 15) == 0;
  constexpr int kEach = MT * NT * 64;
  const int threads = ALL ? 64 * (kSlices / SPW) : (int)blockDim.x;
  auto sum_at = [&](int at, int m, int place) {                        // four weight rows' sums of row m, the first at `place`
    f32x4 pair[kSlices / 2];
#pragma unroll
    for (int i = 0; i < kSlices / 2; ++i) {
      pair[i] = f32x4{0.f, 0.f, 0.f, 0.f};                             // (slices past K are zeros that nobody makes)
      if (!ALL && 2 * i * g.slice >= g.K) continue;
      pair[i] = parts[(SPW == 2 ? i : 2 * i) * kEach + at];
      if (SPW == 1 && (ALL || (2 * i + 1) * g.slice < g.K)) pair[i] += parts[(2 * i + 1) * kEach + at];
    }
    f32x4 sum = ((pair[0] + pair[1]) + (pair[2] + pair[3])) + ((pair[4] + pair[5]) + (pair[6] + pair[7]));
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (!finite(sum[j])) sum[j] = plain_product(A + (size_t)m * g.lda, W + (size_t)weight_row<EPI>(g, place + j) * g.ldw, g.K);
    return sum;
  };
  auto write_four = [&](float* c, f32x4 x, int n, int N) {             // columns n .. n + 3 of N
    if (wide && n + 4 <= N) {
      *reinterpret_cast<f32x4*>(c) = x;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (n + j < N) c[j] = x[j];
    }
  };
  for (int at = tid; at < kEach; at += threads) {
    const int tile = at >> 6, m = m0 + 16 * (tile / NT) + (at & 15), q = (at & 63) >> 4, place = n0 + 16 * (tile % NT) + 4 * q;
    if (m >= g.M) continue;
    if (EPI == FG_PLAIN) {
      if (place < g.N) write_four(C + (size_t)m * g.ldc + place, sum_at(at, m, place), place, g.N);
      continue;
    }
    const int one = (place >> 4) * 8 + 4 * q;                          // of the first kind; the partners are two quads on
    if (q >= 2 || one >= g.N / 2) continue;
    f32x4 x = sum_at(at, m, place), y = sum_at(at + 32, m, place + 8);
    if (EPI == FG_GATED) {
#pragma unroll
      for (int j = 0; j < 4; ++j) x[j] = gate_activation(x[j], g.activation) * y[j];
      write_four(C + (size_t)m * g.ldc + one, x, one, g.N / 2);
    } else {
      const int half = g.head_dim / 2, head = one / half, e = one - head * half;
      if (head < g.num_heads + g.num_kv_heads && g.cos_table) {
        const size_t turn_at = (size_t)g.positions[m] * half + e;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          float lo, hi;
          rotate_pair(x[j], y[j], g.cos_table[turn_at + j], g.sin_table[turn_at + j], lo, hi);
          x[j] = lo;
          y[j] = hi;
        }
      }
      const int slot = head < g.num_heads ? 0 : g.slots[m];
      if (slot < 0) continue;
      const int page = slot / g.block_size, off = slot - page * g.block_size;
      if (head < g.num_heads + g.num_kv_heads) {
        float* c = head < g.num_heads ? C + (size_t)m * g.ldc + (size_t)head * g.head_dim + e
                                      : g.k_pages + (((size_t)page * g.num_kv_heads + (head - g.num_heads)) * g.block_size + off) * g.head_dim + e;
        *reinterpret_cast<f32x4*>(c) = x;
        *reinterpret_cast<f32x4*>(c + half) = y;
      } else {                                                         // values stand transposed in their page
        float* c = g.v_pages + (((size_t)page * g.num_kv_heads + (head - g.num_heads - g.num_kv_heads)) * g.head_dim + e) * g.block_size + off;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          c[(size_t)j * g.block_size] = x[j];
          c[(size_t)(j + half) * g.block_size] = y[j];
        }
      }
    }
  }
}

template <int MT, int NT, int SPW, int PER_SIMD, int EPI>
static int launch_float_gemm(const FloatGemm& g, int batch, bool vec, hipStream_t stream) {
  FloatGemm p = g;
  p.row_tiles = (g.M + 16 * MT - 1) / (16 * MT);
  p.col_tiles = (g.N + 16 * NT - 1) / (16 * NT);
  const int used = (g.K + g.slice - 1) / g.slice, waves = (used + SPW - 1) / SPW;     // wavefronts that have columns: 1 to kSlices / SPW
  const size_t sums = (size_t)waves * MT * NT * 64 * sizeof(f32x4), turns = (size_t)waves * 8 * 272;
  const size_t lds = SPW == 2 ? (size_t)kSlices / SPW * 8 * 272 + sums : (sums > turns ? sums : turns);
  auto kernel = used == kSlices ? gemm_float_kernel<MT, NT, SPW, PER_SIMD, EPI, true, true> : gemm_float_kernel<MT, NT, SPW, PER_SIMD, EPI, true, false>;
  if constexpr (EPI == FG_PLAIN) {
    if (!vec) kernel = used == kSlices ? gemm_float_kernel<MT, NT, SPW, PER_SIMD, EPI, false, true> : gemm_float_kernel<MT, NT, SPW, PER_SIMD, EPI, false, false>;
  }
  if (lds > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return (int)e;
  }
  const dim3 grid((unsigned)(p.col_tiles * p.row_tiles), batch), block(64 * waves);
  hipLaunchKernelGGL(kernel, grid, block, lds, stream, p);
  PLLM_RETURN_LAST_ERROR();
}

template <int EPI>
static int launch_tile(const FloatGemm& g, int batch, bool vec, int rows_tile, int cols_tile, hipStream_t stream) {
  switch (rows_tile * 10 + cols_tile) {
    case 11: return launch_float_gemm<1, 1, 1, 4, EPI>(g, batch, vec, stream);
    case 12: return launch_float_gemm<1, 2, 1, 4, EPI>(g, batch, vec, stream);
    case 22: return launch_float_gemm<2, 2, 1, 4, EPI>(g, batch, vec, stream);
    case 34: return launch_float_gemm<3, 4, 2, 2, EPI>(g, batch, vec, stream);
    case 44: return launch_float_gemm<4, 4, 2, 2, EPI>(g, batch, vec, stream);
    default: return -3;
  }
}

static bool sixteen_bytes(const void* p, long a, long b) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0 && a % 4 == 0 && b % 4 == 0; }

// `batch` products at once, operand b at its base plus b times its batch stride (elements).  `rows_tile`, `cols_tile`: the
// tile in sixteens of rows and weight rows, one of the forms above.
PLLM_API int pllm_gemm_float(const float* A, int lda, long a_batch, const float* W, int ldw, long w_batch, float* C, int ldc, long c_batch,
                             int M, int N, int K, int batch, int rows_tile, int cols_tile, hipStream_t stream) {
  if (M <= 0 || N <= 0 || batch <= 0) return 0;
  if (K <= 0 || batch > 65535) return -2;
  const FloatGemm g{A, W, C, a_batch, w_batch, c_batch, lda, ldw, ldc, M, N, K, slice_columns(K), 0, 0, 0, 0, 0, 0, 0, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
  return launch_tile<FG_PLAIN>(g, batch, K % 4 == 0 && sixteen_bytes(A, lda, a_batch) && sixteen_bytes(W, ldw, w_batch), rows_tile, cols_tile, stream);
}

// One product with something behind it (FG_GATED, FG_ROPE_KV above); rows that 16-byte loads can take.  N: the weight rows.
PLLM_API int pllm_gemm_float_fused(int epi, const float* A, int lda, const float* W, int ldw, float* C, int ldc, int M, int N, int K, int rows_tile,
                                   int cols_tile, int activation, const int* positions, const float* cos_table, const float* sin_table, const int* slots,
                                   float* k_pages, float* v_pages, int num_heads, int num_kv_heads, int head_dim, int block_size, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || K % 4 || N % 2 || !sixteen_bytes(A, lda, 0) || !sixteen_bytes(W, ldw, 0)) return -2;
  const FloatGemm g{A, W, C, 0, 0, 0, lda, ldw, ldc, M, N, K, slice_columns(K), 0, 0, activation, num_heads, num_kv_heads, head_dim, block_size,
                    positions, slots, cos_table, sin_table, k_pages, v_pages};
  if (epi == FG_GATED) return activation >= 0 && activation < PLLM_ACT_COUNT ? launch_tile<FG_GATED>(g, 1, true, rows_tile, cols_tile, stream) : -2;
  if (epi != FG_ROPE_KV) return -3;
  if (head_dim <= 0 || head_dim % 16 || block_size <= 0 || N != (num_heads + 2 * num_kv_heads) * head_dim || !sixteen_bytes(C, ldc, 0) || !sixteen_bytes(k_pages, 0, 0)) return -2;
  return launch_tile<FG_ROPE_KV>(g, 1, true, rows_tile, cols_tile, stream);
}
