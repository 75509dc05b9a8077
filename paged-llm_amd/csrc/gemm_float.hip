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
//     32 (2048 weight rows are 128 workgroups) and few enough registers for two workgroups on a compute unit: 8 rows x 2048 x 2048 in 7.0
//     us (8.5 with the float instruction, which takes the weights' loads in operand order as well), 11264 x 2048 in 18.4 (23.4), 2048 x
//     5632 in 14.4 (18.6); 64 rows x 2048 x 2048 in 10.1 (13.4).
//     There the split is what bounds the smaller ones (half of a wavefront's vector instructions are the rows', half the weights'; more
//     loads under way, two to four steps, made every one of them slower), and 128 workgroups leave half of the compute units idle: where the reader adds
//     two sums, two workgroups take eight slices each (pllm_gemm_float_halves: 8 rows x 2048 x 2048 8.1 -> 6.4 us, x 5632 19.0 -> 13.5 with weights
//     from memory).
//   * Many rows: bound by the same way (a tile of 64 x 64 draws 42 bytes a clock at the matrix cores' rate, of 45 that the L2 gives) and
//     by a wavefront's chain of load, turn, split and product.  Eight wavefronts take two slices each, one after the other, with up to 256
//     registers a lane; the first slice's sums wait in LDS.  301 rows x 2048 x 2048 / 5632 in 27 / 64 us (37 / 86 with the float
//     instruction), x 11264 x 2048 in 123 (168), 1024 rows x 2048 x 5632 in 160 (222).
//   * Short K (the matrices of heads): bound by memory and by what a workgroup takes to start and end.  Only the wavefronts that
//     have columns are launched (300 / 1500 rows of 64 heads of 64 x 64: 6.4 / 20 us, with the float instruction 6.0 / 19; one row 3.1 and 2.7).
// Loads need no more than the alignment of a float: K and strides may be any (8 / 301 / 1024 rows x 2048 x 2047 in
// 7.7 / 30.6 / 73 us; 8.9 / 39 / 96 with the float instruction, 10.2 / 36 / 84 element by element).
// Results that are not finite are made again by the whole workgroup, each wavefront its slices of K, in tiles of 16 x 16 (a row of NaN: 8 rows x 2048 x
// 2048 9.7 -> 13.5 us, 301 rows 26 -> 55, 8 rows x 32000 x 2048 51 -> 102).
// Which tile a product takes is the host's choice by the rounds of workgroups (ops.float_gemm_plan, ops.float_split_plan).
//
// SPLIT: with many rows the split was most of a wavefront's vector instructions, and each tile of weights was split again by every workgroup
// of its rows.  A second copy of the weights holds their parts, made once, in operand order: whole kilobytes that go straight to
// the matrix cores.  Of the steady state's 2.3 us a step of two wavefronts (64 x 64, 32 columns each) the products are 1.6 now.  301 rows x 2048 x
// 2048 27.4 -> 24.1 us, x 5632 62.8 -> 52.7, 11264 x 2048 gated 125.6 -> 107.8, 32000 x 2048 313 -> 287; 512 rows x 2048 x 5632 82 -> 70.
#include "float_split.h"

#include <type_traits>

using namespace pllm;

struct FloatGemm {
  const float* A;
  const float* W;
  const bf16x8* W_split;                                               // (SPLIT) the weights' parts, or null
  float* C;
  long a_batch, w_batch, c_batch, c_range;                             // (c_range: from the first range's sums to the second's)
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
// FAR: rows so far apart that an offset inside a tile takes 64 bits.
// SPLIT: the weights' parts come from W_split, as pllm_float_split_weights lays them out.
// RANGES: workgroups of a tile (blockIdx.z), each with as many of the slices, whose sums are results of their own.
template <int MT, int NT, int SPW, int PER_SIMD, int EPI, bool FAR, bool ALL, bool SPLIT, int RANGES>
__global__ __launch_bounds__(64 * (kSlices / SPW / RANGES), PER_SIMD) void gemm_float_kernel(FloatGemm g) {
  static_assert(RANGES == 1 || (RANGES == 2 && SPW == 1 && EPI == FG_PLAIN && ALL), "halves of the tree");
  constexpr int kOwn = kSlices / RANGES;
  const int first_slice = RANGES == 1 ? 0 : (int)blockIdx.z * kOwn;
  constexpr int kPad = 272;                                            // bytes: a chunk of 16 bytes of 16 rows, and 16 against bank conflicts
  extern __shared__ __attribute__((aligned(16))) unsigned char gf_lds[];
  __shared__ unsigned waiting;                                         // the tiles of 16 x 16 with a sum that is not finite
  f32x4* parts = reinterpret_cast<f32x4*>(gf_lds + (SPW == 2 ? kSlices / SPW * 8 * kPad : 0));   // at the end: [wavefronts][MT * NT][64]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, quad = lane >> 4;
  if (tid == 0) waiting = 0;
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
  float* C = g.C + (size_t)blockIdx.y * g.c_batch + (RANGES == 1 ? 0 : (size_t)blockIdx.z * g.c_range);

  // A tile of 16 rows x 32 columns under way: two loads of 8 rows x 128 bytes.
  struct Tile { f32x4 x[2]; };
  using Offset = std::conditional_t<FAR, size_t, unsigned>;
  const int w_first = EPI == FG_PLAIN ? n0 : 0, c8 = 4 * (lane & 7);
  Offset a_at[MT][2], w_at[NT][2];                                     // in elements from the tile's first row; rows past the end repeat the last one
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int r = 8 * j + (lane >> 3);
#pragma unroll
    for (int i = 0; i < MT; ++i) a_at[i][j] = (Offset)min(16 * i + r, g.M - 1 - m0) * g.lda + c8;
#pragma unroll
    for (int i = 0; i < NT; ++i) w_at[i][j] = SPLIT ? 0 : (Offset)(weight_row<EPI>(g, n0 + 16 * i + r) - w_first) * g.ldw + c8;
  }
  const float *a_rows = A + (size_t)m0 * g.lda, *w_rows = W + (size_t)w_first * g.ldw;
  auto load = [&](const float* rows, const Offset* at, int k, bool tail) {   // `tail`: zeros from column K on
    Tile t;
#pragma unroll
    for (int j = 0; j < 2; ++j) t.x[j] = tail ? four_of(rows + k + at[j], g.K - k - c8) : four_of(rows + k + at[j]);
    return t;
  };
  auto operand = [&](const Tile& t) {
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

  const int begin = min((first_slice + wave * SPW) * g.slice, g.K), end = min(begin + SPW * g.slice, g.K);
  const int steps = (end - begin) / kStep, per_slice = g.slice / kStep;  // whole steps; the last slice may have a tail
#pragma unroll
  for (int i = 0; i < MT * NT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto second_slice = [&](int step) {                                  // which starts from zero
    if (SPW != 2 || step + 1 != per_slice) return;
#pragma unroll
    for (int i = 0; i < MT * NT; ++i) {
      own_part[i * 64] = acc[i];
      acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  };
  if constexpr (SPLIT) {
    // The parts of a tile of 16 weight rows are 3 KB for every 32 columns, in operand order; a step's are asked for a step ahead.
    const int all_steps = (g.K + kStep - 1) / kStep, last_tile = (g.N + 15) / 16 - 1;
    const bf16x8* parts_of[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) parts_of[n] = g.W_split + (size_t)min(col_tile * NT + n, last_tile) * all_steps * (3 * 64) + lane;
    auto load_parts = [&](Triple* w, int k) {
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int p = 0; p < 3; ++p) w[n].part[p] = parts_of[n][(size_t)(k / kStep) * (3 * 64) + p * 64];
    };
    if (steps > 0) {
      Tile a[MT];
      Triple w0[NT], w1[NT];
      load_parts(w0, begin);
#pragma unroll
      for (int i = 0; i < MT; ++i) a[i] = load(a_rows, a_at[i], begin, false);
      __builtin_amdgcn_sched_barrier(0);
      auto one_step = [&](const Triple* now, Triple* next, int step) {
        const int k = begin + min(step + 1, steps - 1) * kStep;        // (past the last step: that one again, not used)
        load_parts(next, k);
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          const Triple at = split(operand(a[i]));
          a[i] = load(a_rows, a_at[i], k, false);
          __builtin_amdgcn_sched_barrier(0);
          multiply(now, at, i);
        }
        second_slice(step);
      };
#pragma unroll 1
      for (int step = 0; step + 1 < steps; step += 2) {
        one_step(w0, w1, step);
        one_step(w1, w0, step + 1);
      }
      if (steps & 1) one_step(w0, w1, steps - 1);
    }
    if (begin + steps * kStep < end) {                                 // less than a step is left (the parts past K are zeros)
      const int k = begin + steps * kStep;
      Triple w0[NT];
      load_parts(w0, k);
#pragma unroll
      for (int i = 0; i < MT; ++i) multiply(w0, split(operand(load(a_rows, a_at[i], k, true))), i);
    }
  } else {
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
        second_slice(step);
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
  }
  if (SPW == 1) __syncthreads();                                       // (the sums take the place of the tiles on their way)
#pragma unroll
  for (int i = 0; i < MT * NT; ++i) own_part[i * 64] = SPW == 2 && steps >= per_slice ? own_part[i * 64] + acc[i] : acc[i];
  __syncthreads();

  const bool wide = (g.ldc & 3) == 0 && (reinterpret_cast<uintptr_t>(C) & 15) == 0;
  constexpr int kEach = MT * NT * 64;
  const int threads = ALL ? 64 * (kOwn / SPW) : (int)blockDim.x;
  auto sum_at = [&](int at) {                                          // of a lane's four weight rows and row
    f32x4 pair[kOwn / 2];
#pragma unroll
    for (int i = 0; i < kOwn / 2; ++i) {
      pair[i] = f32x4{0.f, 0.f, 0.f, 0.f};                             // (slices past K are zeros that nobody makes)
      if (!ALL && 2 * i * g.slice >= g.K) continue;
      pair[i] = parts[(SPW == 2 ? i : 2 * i) * kEach + at];
      if (SPW == 1 && (ALL || (2 * i + 1) * g.slice < g.K)) pair[i] += parts[(2 * i + 1) * kEach + at];
    }
    const f32x4 half = (pair[0] + pair[1]) + (pair[2] + pair[3]);
    if constexpr (RANGES == 2) return half;
    else return half + ((pair[4] + pair[5]) + (pair[6] + pair[7]));
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
  auto finish = [&](int at, f32x4 x) {                                 // what stands behind the sums; by whole wavefronts, a tile of 16 x 16 each
    const int tile = at >> 6, q = (at & 63) >> 4, m = m0 + 16 * (tile / NT) + (at & 15), place = n0 + 16 * (tile % NT) + 4 * q;
    if (EPI == FG_PLAIN) {
      if (m < g.M && place < g.N) write_four(C + (size_t)m * g.ldc + place, x, place, g.N);
      return;
    }
    f32x4 y;                                                           // of lanes 0 to 31: the partners' sums
#pragma unroll
    for (int j = 0; j < 4; ++j) y[j] = __shfl_xor(x[j], 32);
    const int one = (place >> 4) * 8 + 4 * q;                          // of the first kind; the partners are two quads on
    if (m >= g.M || q >= 2 || one >= g.N / 2) return;
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
      if (slot < 0) return;
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
  };
  auto fine = [](f32x4 x) { return __all(finite(x[0]) && finite(x[1]) && finite(x[2]) && finite(x[3])); };
  f32x4* kept = SPW == 2 ? reinterpret_cast<f32x4*>(gf_lds) : parts + (threads >> 6) * kEach;   // tiles with a sum that is not finite wait here
  for (int at = tid; at < kEach; at += threads) {
    const f32x4 x = sum_at(at);
    if (fine(x)) {
      finish(at, unscaled(x));
    } else {
      kept[at] = x;
      if (lane == 0) atomicOr(&waiting, 1u << (at >> 6));
    }
  }
  __syncthreads();
  const unsigned tiles = __builtin_amdgcn_readfirstlane(waiting);
  if (tiles == 0) return;
#pragma unroll 1
  for (int i = 0; i < MT * NT; ++i) {                                  // (each wavefront its slices)
    if (!(tiles >> i & 1)) continue;
    const float *a = A + (size_t)min(m0 + 16 * (i / NT) + r16, g.M - 1) * g.lda, *w = W + (size_t)weight_row<EPI>(g, n0 + 16 * (i % NT) + r16) * g.ldw;
    f32x4 sum{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int s = wave * SPW; s < wave * SPW + SPW; ++s) {
      const f32x4 x = plain_sums(a, w, min((first_slice + s) * g.slice, g.K), min((first_slice + s + 1) * g.slice, g.K));
      sum = s == wave * SPW ? x : sum + x;
    }
    own_part[i * 64] = sum;
  }
  __syncthreads();
  for (int at = tid; at < kEach; at += threads) {
    if (!(tiles >> (at >> 6) & 1)) continue;
    const f32x4 split_sum = kept[at], plain = sum_at(at);
    f32x4 x = unscaled(split_sum);
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = finite(split_sum[j]) ? x[j] : plain[j];
    finish(at, x);
  }
}

template <int MT, int NT, int SPW, int PER_SIMD, int EPI, bool SPLIT = false, int RANGES = 1>
static int launch_float_gemm(const FloatGemm& g, int batch, bool far, hipStream_t stream) {
  FloatGemm p = g;
  p.row_tiles = (g.M + 16 * MT - 1) / (16 * MT);
  p.col_tiles = (g.N + 16 * NT - 1) / (16 * NT);
  const int used = (g.K + g.slice - 1) / g.slice, waves = (used / RANGES + SPW - 1) / SPW;   // wavefronts that have columns: 1 to kSlices / SPW
  if (RANGES > 1 && used != kSlices) return -2;
  const size_t sums = (size_t)waves * MT * NT * 64 * sizeof(f32x4), turns = (size_t)waves * 8 * 272;
  const size_t kept = (size_t)MT * NT * 64 * sizeof(f32x4);                            // (SPW = 2: in the place of the tiles on their way)
  const size_t lds = SPW == 2 ? (size_t)kSlices / SPW * 8 * 272 + sums : (sums + kept > turns ? sums + kept : turns);
  static_assert(SPW == 1 || MT * NT * 64 * sizeof(f32x4) <= kSlices / SPW * 8 * 272, "the tiles that wait fit there");
  constexpr int kFewer = SPW == 1 ? 4 : PER_SIMD;                      // (workgroups of fewer wavefronts)
  auto kernel = gemm_float_kernel<MT, NT, SPW, PER_SIMD, EPI, false, true, SPLIT, RANGES>;
  if constexpr (RANGES == 1) {
    if (used != kSlices) kernel = gemm_float_kernel<MT, NT, SPW, kFewer, EPI, false, false, SPLIT, 1>;
  }
  if constexpr (EPI == FG_PLAIN && !SPLIT && RANGES == 1) {
    if (far) kernel = used == kSlices ? gemm_float_kernel<MT, NT, SPW, PER_SIMD, EPI, true, true, false, 1> : gemm_float_kernel<MT, NT, SPW, kFewer, EPI, true, false, false, 1>;
  }
  if (lds > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return (int)e;
  }
  const dim3 grid((unsigned)(p.col_tiles * p.row_tiles), batch, RANGES), block(64 * waves);
  hipLaunchKernelGGL(kernel, grid, block, lds, stream, p);
  PLLM_RETURN_LAST_ERROR();
}

template <int EPI>
static int launch_tile(const FloatGemm& g, int batch, bool far, int rows_tile, int cols_tile, hipStream_t stream) {
  switch (rows_tile * 10 + cols_tile) {
    case 11: return launch_float_gemm<1, 1, 1, 8, EPI>(g, batch, far, stream);
    case 12: return launch_float_gemm<1, 2, 1, 4, EPI>(g, batch, far, stream);
    case 22: return launch_float_gemm<2, 2, 1, 4, EPI>(g, batch, far, stream);
    case 34: return launch_float_gemm<3, 4, 2, 2, EPI>(g, batch, far, stream);
    case 44: return launch_float_gemm<4, 4, 2, 2, EPI>(g, batch, far, stream);
    default: return -3;
  }
}

static bool far(int lda, int ldw) { return lda > 1 << 26 || ldw > 1 << 26; }      // (64 rows within 2^32 elements)
static bool sixteen_bytes(const void* p, long a, long b) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0 && a % 4 == 0 && b % 4 == 0; }

// `batch` products at once, operand b at its base plus b times its batch stride (elements).  `rows_tile`, `cols_tile`: the
// tile in sixteens of rows and weight rows, one of the forms above.
PLLM_API int pllm_gemm_float(const float* A, int lda, long a_batch, const float* W, int ldw, long w_batch, float* C, int ldc, long c_batch,
                             int M, int N, int K, int batch, int rows_tile, int cols_tile, hipStream_t stream) {
  if (M <= 0 || N <= 0 || batch <= 0) return 0;
  if (K <= 0 || batch > 65535) return -2;
  const FloatGemm g{A, W, nullptr, C, a_batch, w_batch, c_batch, 0, lda, ldw, ldc, M, N, K, slice_columns(K), 0, 0, 0, 0, 0, 0, 0, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
  return launch_tile<FG_PLAIN>(g, batch, far(lda, ldw), rows_tile, cols_tile, stream);
}

// The same product of few rows as two sums, C [2][M][N]: of the first and of the last eight slices, whose sum is the result (K with columns in all
// sixteen, rows and weight rows within 32-bit offsets of a tile).
PLLM_API int pllm_gemm_float_halves(const float* A, int lda, const float* W, int ldw, float* C, int M, int N, int K, int cols_tile, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || far(lda, ldw)) return -2;
  const FloatGemm g{A, W, nullptr, C, 0, 0, 0, (long)M * N, lda, ldw, N, M, N, K, slice_columns(K), 0, 0, 0, 0, 0, 0, 0, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
  return cols_tile == 1 ? launch_float_gemm<1, 1, 1, 4, FG_PLAIN, false, 2>(g, 1, false, stream) : launch_float_gemm<1, 2, 1, 4, FG_PLAIN, false, 2>(g, 1, false, stream);
}

template <int EPI>
static int launch_split_tile(const FloatGemm& g, int rows_tile, int cols_tile, hipStream_t stream) {
  switch (rows_tile * 10 + cols_tile) {
    case 24: return launch_float_gemm<2, 4, 2, 2, EPI, true>(g, 1, false, stream);
    case 34: return launch_float_gemm<3, 4, 2, 2, EPI, true>(g, 1, false, stream);
    case 44: return launch_float_gemm<4, 4, 2, 2, EPI, true>(g, 1, false, stream);
    default: return -3;
  }
}

// One product (FG_PLAIN), or one with something behind it (FG_GATED, FG_ROPE_KV above); all weight rows within 2^32 elements.  N: the
// weight rows.  W_split: the weights' parts in the order that this product takes them, or null; with them the tile is one of those above.
PLLM_API int pllm_gemm_float_fused(int epi, const float* A, int lda, const float* W, int ldw, const void* W_split, float* C, int ldc, int M, int N, int K,
                                   int rows_tile, int cols_tile, int activation, const int* positions, const float* cos_table, const float* sin_table,
                                   const int* slots, float* k_pages, float* v_pages, int num_heads, int num_kv_heads, int head_dim, int block_size,
                                   hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || far(lda, 0) || (long)N * ldw > 1l << 32 || reinterpret_cast<uintptr_t>(W_split) % 16) return -2;
  const FloatGemm g{A, W, (const bf16x8*)W_split, C, 0, 0, 0, 0, lda, ldw, ldc, M, N, K, slice_columns(K), 0, 0, activation, num_heads, num_kv_heads, head_dim,
                    block_size, positions, slots, cos_table, sin_table, k_pages, v_pages};
  if (epi == FG_PLAIN) return W_split ? launch_split_tile<FG_PLAIN>(g, rows_tile, cols_tile, stream) : -3;
  if (N % 2) return -2;
  if (epi == FG_GATED) {
    if (activation < 0 || activation >= PLLM_ACT_COUNT) return -2;
    return W_split ? launch_split_tile<FG_GATED>(g, rows_tile, cols_tile, stream) : launch_tile<FG_GATED>(g, 1, false, rows_tile, cols_tile, stream);
  }
  if (epi != FG_ROPE_KV) return -3;
  if (head_dim <= 0 || head_dim % 16 || block_size <= 0 || N != (num_heads + 2 * num_kv_heads) * head_dim || !sixteen_bytes(C, ldc, 0) || !sixteen_bytes(k_pages, 0, 0)) return -2;
  return W_split ? launch_split_tile<FG_ROPE_KV>(g, rows_tile, cols_tile, stream) : launch_tile<FG_ROPE_KV>(g, 1, false, rows_tile, cols_tile, stream);
}

// The parts of a matrix's floats in the order in which a product with this epilogue takes them:
// [tiles of 16 weight rows][steps of 32 columns][3 parts][64 lanes][8], zeros past column K.
template <int EPI>
__global__ __launch_bounds__(64) void float_split_weights_kernel(FloatGemm g, bf16x8* out) {
  const int lane = threadIdx.x, k = blockIdx.x * kStep + 4 * (lane >> 4);
  for (int tile = blockIdx.y; tile < g.col_tiles; tile += gridDim.y) {   // (a grid has 65,535 of them at most)
    const float* row = g.W + (size_t)weight_row<EPI>(g, 16 * tile + (lane & 15)) * g.ldw + k;
    const Triple t = split(Octet{four_of(row, g.K - k), four_of(row + 16, g.K - k - 16)});
#pragma unroll
    for (int p = 0; p < 3; ++p) out[(((size_t)tile * gridDim.x + blockIdx.x) * 3 + p) * 64 + lane] = t.part[p];
  }
}

PLLM_API int pllm_float_split_weights(int epi, const float* W, int ldw, int N, int K, int head_dim, void* out, hipStream_t stream) {
  if (N <= 0 || N > 0x7fffffff - 15 || K <= 0 || reinterpret_cast<uintptr_t>(out) % 16) return -2;
  if ((epi == FG_GATED && N % 2) || (epi == FG_ROPE_KV && (head_dim <= 0 || head_dim % 16 || N % head_dim))) return -2;
  FloatGemm g{};
  g.W = W; g.ldw = ldw; g.N = N; g.K = K; g.head_dim = head_dim; g.col_tiles = (N + 15) / 16;
  auto kernel = epi == FG_PLAIN ? float_split_weights_kernel<FG_PLAIN> : epi == FG_GATED ? float_split_weights_kernel<FG_GATED> : float_split_weights_kernel<FG_ROPE_KV>;
  hipLaunchKernelGGL(kernel, dim3((K + kStep - 1) / kStep, min(g.col_tiles, 65535)), dim3(64), 0, stream, g, (bf16x8*)out);
  PLLM_RETURN_LAST_ERROR();
}
