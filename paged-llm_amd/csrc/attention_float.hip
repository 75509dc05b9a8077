// Paged causal attention of the true 32-bit path on the float matrix cores (v_mfma_f32_16x16x4_f32, exponentials and sums
// in float): head sizes that are multiples of 16 up to 256, pages whose size is a multiple of 16 positions.  The arrays,
// masks, score terms and weightings are those of attention_generic.hip, which keeps every other shape.
//
// A workgroup owns 16 columns, a column being a (query token, query head) pair of one sequence and one kv head, so that the
// heads of a group share every key and value that is loaded.  S^T = K Q^T leaves a lane with four keys of one column, which
// is the operand layout of O^T = V^T P^T as it stands: a lane's 16-byte load of V (four consecutive positions of a channel)
// meets its four weights in four instructions, and nothing is moved between lanes.
//
// The keys are cut into blocks of 64 at absolute positions 0, 64, 128, ...; wavefront w of the workgroup's eight (fewer for
// heads above 128 and short windows) takes the blocks whose number is w modulo their count, each with a running maximum of its own,
// and the wavefronts' results are joined in their order.  A block that a column does not see changes none of its bits, so a
// column's result is the same however the tokens were cut into steps or batched.  Of a block that is seen in part, the tiles of 16
// keys that no column sees are left out (a prompt of 17 tokens, 32 heads of 64 on 4: 12.5 us, 13.5 with the whole block; 24 heads of
// 256 on 8: 19 and 27).
//
// What bounds it: a wavefront's chain of load, scores, exponentials and values per block for few columns (decoding: 8
// requests, contexts to 700, 32 heads of 64 on 4: 186 us with one wavefront per token and head), and the matrix cores
// beside the L2 for prompts (301 tokens, the same heads: 253 us before).
#include "common.h"

using namespace pllm;

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kColumns = 16, kBlock = 64, kTile = 16, kTiles = kBlock / kTile;

struct FloatAttention {
  const float *q, *k_pages, *v_pages;
  float* out;
  const int *block_tables, *cu_seqlens_q, *seq_lens_k;
  const float* head_bias;
  ScoreTerms terms;
  int q_stride, out_stride, bt_stride, num_seqs, num_heads, num_kv_heads, block_size, window, keep_first, weighting;
  float scale;
};

// Sums and maxima over the four lanes that hold a column (l, l + 16, l + 32, l + 48).
__device__ __forceinline__ float column_max(float v) {
  v = fmaxf(v, __shfl_xor(v, 16));
  return fmaxf(v, __shfl_xor(v, 32));
}
__device__ __forceinline__ float column_sum(float v) {
  v += __shfl_xor(v, 16);
  return v + __shfl_xor(v, 32);
}

// DT: head size / 16.
template <int DT, int WAVES>
__global__ __launch_bounds__(64 * WAVES, DT <= 8 ? 2 : 1) void paged_attention_float_kernel(FloatAttention p) {
  constexpr int D = 16 * DT, kChunk = DT < 8 ? DT : 8;
  constexpr bool kEarly = DT <= 4;                                     // registers for a whole block's keys and values at once
  __shared__ float lds_m[WAVES][kColumns], lds_l[WAVES][kColumns];
  extern __shared__ __attribute__((aligned(16))) unsigned char fa_lds[];
  f32x4* lds_o = reinterpret_cast<f32x4*>(fa_lds);                     // [WAVES][DT][64]
  const int tid = threadIdx.x, lane = tid & 63, column = lane & 15, quad = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = p.num_heads / p.num_kv_heads, kvh = blockIdx.y;

  // Sequence s has the tiles from floor(cu[s] group / 16) + s on; those that its columns do not fill end at once.
  int lo = 0, hi = p.num_seqs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if ((int)((long)p.cu_seqlens_q[mid] * group / kColumns) + mid <= (int)blockIdx.x) lo = mid; else hi = mid - 1;
  }
  const int seq = lo, q_begin = p.cu_seqlens_q[seq], num_q = p.cu_seqlens_q[seq + 1] - q_begin;
  const int first_column = ((int)blockIdx.x - ((int)((long)q_begin * group / kColumns) + seq)) * kColumns;
  const long columns = (long)num_q * group;
  if (first_column >= columns) return;
  const int len_k = p.seq_lens_k[seq];
  const int* bt = p.block_tables + (size_t)seq * p.bt_stride;
  const int last_column = (int)min((long)first_column + kColumns, columns) - 1;
  const int c = min(first_column + column, last_column);               // (columns past the end repeat the last one)
  const int tok = q_begin + c / group, head = kvh * group + c % group, pos = len_k - num_q + c / group;
  const int first_key = first_visible_key(pos, p.window);
  const int pos_max = len_k - num_q + last_column / group, pos_min = len_k - num_q + first_column / group;
  const int any_from = first_visible_key(pos_min, p.window);           // keys that some column sees: from here to pos_max, and the kept ones
  const int all_from = first_visible_key(pos_max, p.window);           // ... that every column sees: from here to pos_min

  f32x4 q[DT];
  {
    const float* row = p.q + (size_t)tok * p.q_stride + (size_t)head * D + 4 * quad;
#pragma unroll
    for (int t = 0; t < DT; ++t) q[t] = *reinterpret_cast<const f32x4*>(row + 16 * t);
  }
  const bool softmax = p.weighting == 0;
  const float slope = p.terms.slopes ? p.terms.slopes[head] : 0.f;
  const float bias = !softmax && p.head_bias ? p.head_bias[head] : 0.f;
  float m = -INFINITY, l = 0.f;                                        // l: this lane's share of the column's sum
  if (p.terms.sinks && softmax && wave == 0) {                         // as if one key with this score and no value had been seen
    m = p.terms.sinks[head];
    l = quad == 0 ? 1.f : 0.f;
  }
  f32x4 o[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int b = wave; b * kBlock <= pos_max; b += WAVES) {
    const int n0 = b * kBlock;
    if (n0 + kBlock - 1 < any_from && n0 >= p.keep_first) {            // between the kept positions and the window: on to the window's first
      const int skip = any_from / kBlock - b;
      b += (skip + WAVES - 1) / WAVES * WAVES - WAVES;
      continue;
    }
    const bool whole = n0 + kBlock - 1 <= pos_min && n0 >= all_from;   // every column sees every key of the block
    f32x4 s[kTiles];
    bool live[kTiles], all_live = true;                                // (the same for all lanes: a tile that no column sees is left out)
    const float *k_at[kTiles], *v_at[kTiles];                          // (a tile lies inside one page)
#pragma unroll
    for (int i = 0; i < kTiles; ++i) {
      const int n = n0 + i * kTile;
      live[i] = n <= pos_max && (n + kTile > any_from || n < p.keep_first);
      all_live = all_live && live[i];
      const int from = live[i] ? n : pos_max / kTile * kTile;          // (a tile that no column sees: any valid one, for loads without conditions)
      const size_t page = (size_t)bt[from / p.block_size] * p.num_kv_heads + kvh;
      k_at[i] = p.k_pages + (page * p.block_size + from % p.block_size + column) * D + 4 * quad;
      v_at[i] = p.v_pages + (page * D + column) * p.block_size + from % p.block_size + 4 * quad;
    }
    f32x4 v_early[kEarly ? kTiles : 1][kEarly ? DT : 1];
    if (kEarly) {
      f32x4 k[kTiles][DT <= 4 ? DT : 1];
#pragma unroll
      for (int i = 0; i < kTiles; ++i)
#pragma unroll
        for (int t = 0; t < DT; ++t) k[i][t] = *reinterpret_cast<const f32x4*>(k_at[i] + 16 * t);
#pragma unroll
      for (int i = 0; i < kTiles; ++i)
#pragma unroll
        for (int t = 0; t < DT; ++t) v_early[i][t] = *reinterpret_cast<const f32x4*>(v_at[i] + (size_t)16 * t * p.block_size);
#pragma unroll
      for (int i = 0; i < kTiles; ++i) s[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (all_live) {
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < kTiles; ++i) s[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i][t][j], q[t][j], s[i], 0, 0, 0);
      } else {
#pragma unroll
        for (int i = 0; i < kTiles; ++i)
          if (live[i]) {
#pragma unroll
            for (int t = 0; t < DT; ++t)
#pragma unroll
              for (int j = 0; j < 4; ++j) s[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i][t][j], q[t][j], s[i], 0, 0, 0);
          }
      }
    } else {
#pragma unroll
      for (int i = 0; i < kTiles; ++i) {
        s[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (!live[i]) continue;
#pragma unroll
        for (int t0 = 0; t0 < DT; t0 += kChunk) {
          f32x4 k[kChunk];
#pragma unroll
          for (int t = 0; t < kChunk; ++t)
            if (t0 + t < DT) k[t] = *reinterpret_cast<const f32x4*>(k_at[i] + 16 * (t0 + t));
#pragma unroll
          for (int t = 0; t < kChunk; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j)
              if (t0 + t < DT) s[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[t][j], q[t0 + t][j], s[i], 0, 0, 0);
        }
      }
    }
    float alpha = 1.f;
    auto seen = [&](int n) { return whole || (n <= pos && (n >= first_key || n < p.keep_first)); };
#pragma unroll
    for (int i = 0; i < kTiles; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int n = n0 + i * kTile + 4 * quad + j;
        float x = capped_score(s[i][j] * p.scale, p.terms.cap);
        if (p.terms.slopes) x += slope * (float)(n - pos);
        if (softmax) s[i][j] = seen(n) ? x : -INFINITY;
        else s[i][j] = seen(n) ? 1.f / (1.f + expf(-(x + bias))) : 0.f;
      }
    if (softmax) {
      float top = m;
#pragma unroll
      for (int i = 0; i < kTiles; ++i) top = fmaxf(top, fmaxf(fmaxf(s[i][0], s[i][1]), fmaxf(s[i][2], s[i][3])));
      top = column_max(top);
      const float from = top == -INFINITY ? 0.f : top;                 // (a column that has seen no key yet)
      alpha = expf(m - from);
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < kTiles; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          s[i][j] = expf(s[i][j] - from);
          sum += s[i][j];
        }
      m = top;
      l = l * alpha + sum;
#pragma unroll
      for (int t = 0; t < DT; ++t) o[t] *= alpha;
    }
#pragma unroll
    for (int i = 0; i < kTiles; ++i) {
      if (!live[i]) continue;
#pragma unroll
      for (int t0 = 0; t0 < DT; t0 += kChunk) {
        const int n = n0 + i * kTile;
        f32x4 v[kChunk];
#pragma unroll
        for (int t = 0; t < kChunk; ++t)
          if (t0 + t < DT) v[t] = kEarly ? v_early[kEarly ? i : 0][kEarly ? t0 + t : 0] : *reinterpret_cast<const f32x4*>(v_at[i] + (size_t)16 * (t0 + t) * p.block_size);
        if (!whole) {
          // A weight of zero must not meet a value that is no number: slots that no column sees hold anything (zeros
          // instead), and a value that is not finite is left out here and given to the columns that see it, one by one.
          bool odd = false;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int key = n + 4 * quad + j;
            const bool any = key <= pos_max && (key >= any_from || key < p.keep_first);
#pragma unroll
            for (int t = 0; t < kChunk; ++t)
              if (t0 + t < DT) {
                const bool finite = fabsf(v[t][j]) < INFINITY;
                odd = odd || (any && !finite);
                v[t][j] = any && finite ? v[t][j] : 0.f;
              }
          }
          if (__any(odd)) {
            const float* at = v_at[i] + (4 * quad - column) * p.block_size - 4 * quad;
#pragma unroll 1
            for (int key = 0; key < kTile; ++key) {
              const float own = key % 4 == 0 ? s[i][0] : key % 4 == 1 ? s[i][1] : key % 4 == 2 ? s[i][2] : s[i][3];
              const float weight = __shfl(own, (key / 4) * 16 + column);
              if (n + key > pos_max || !seen(n + key)) continue;
#pragma unroll
              for (int t = 0; t < kChunk; ++t)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                  if (t0 + t < DT) {
                    const float x = at[(size_t)(16 * (t0 + t) + j) * p.block_size + key];
                    if (!(fabsf(x) < INFINITY)) o[t0 + t][j] = fmaf(weight, x, o[t0 + t][j]);
                  }
            }
          }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int t = 0; t < kChunk; ++t)
            if (t0 + t < DT) o[t0 + t] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[t][j], s[i][j], o[t0 + t], 0, 0, 0);
      }
    }
  }

  l = column_sum(l);
  if (quad == 0) {
    lds_m[wave][column] = m;
    lds_l[wave][column] = l;
  }
#pragma unroll
  for (int t = 0; t < DT; ++t) lds_o[(wave * DT + t) * 64 + lane] = o[t];
  __syncthreads();
  if (first_column + column > last_column) return;
  float factor[WAVES], inv = 1.f;
  if (softmax) {
    float top = lds_m[0][column], sum = 0.f;
#pragma unroll
    for (int w = 1; w < WAVES; ++w) top = fmaxf(top, lds_m[w][column]);
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      factor[w] = expf(lds_m[w][column] - top);                        // (finite: a query sees itself)
      sum += lds_l[w][column] * factor[w];
    }
    inv = 1.f / sum;
  }
  for (int t = wave; t < DT; t += WAVES) {
    f32x4 sum = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const f32x4 part = lds_o[(w * DT + t) * 64 + lane];
      sum = softmax ? sum + part * factor[w] : sum + part;
    }
    *reinterpret_cast<f32x4*>(p.out + (size_t)tok * p.out_stride + (size_t)head * D + 16 * t + 4 * quad) = sum * inv;
  }
}

// Wavefronts of a workgroup: eight (heads above 128: four), or one or two for layers whose window is so short that a tile of columns sees
// keys of two to four blocks only.  Further wavefronts would find no block, and keep other workgroups off the compute unit (200
// requests at context 300, 16 heads of 64: a window of 30 31 us with one wavefront and 69 with four, a window of 100 51 us with two,
// 78 with four and 135 with eight, where the plain kernel takes 28 and 66; one request 12 to 16 us in any form).  The window is the
// layer's, so a layer's columns keep their order of additions in every step.  (Relative error against 64 bits with eight wavefronts /
// as now / in the plain kernel, 700 positions: window 30 3.28e-7 / 3.29e-7 / 3.27e-7, 100 4.38e-7 / 4.38e-7 / 4.50e-7; one
// wavefront at 64 would have 4.10e-7 against 4.03e-7.)
constexpr int kOneWaveWindow = 32, kTwoWaveWindow = 128;

template <int DT, int kWaves>
static int launch_float_attention(const FloatAttention& p, int total_q, hipStream_t stream) {
  const int group = p.num_heads / p.num_kv_heads;
  const dim3 grid((unsigned)((long)total_q * group / kColumns + p.num_seqs), p.num_kv_heads), block(64 * kWaves);
  const size_t lds = (size_t)kWaves * DT * 64 * sizeof(f32x4);
  if (lds > 48 * 1024) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(paged_attention_float_kernel<DT, kWaves>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return (int)e;
  }
  hipLaunchKernelGGL((paged_attention_float_kernel<DT, kWaves>), grid, block, lds, stream, p);
  PLLM_RETURN_LAST_ERROR();
}

PLLM_API int pllm_paged_attention_float(const float* q, int q_stride, const float* k_pages, const float* v_pages, float* out, int out_stride,
                                        const int* block_tables, int bt_stride, const int* cu_seqlens_q, const int* seq_lens_k, int num_seqs,
                                        int total_q, int num_heads, int num_kv_heads, int head_dim, int block_size, float scale, int window,
                                        float score_cap, const float* slopes, const float* sinks, int keep_first, int weighting,
                                        const float* head_bias, hipStream_t stream) {
  if (total_q <= 0 || num_seqs <= 0) return 0;
  if (head_dim <= 0 || head_dim % 16 || head_dim > 256 || block_size <= 0 || block_size % kTile) return -2;
  if (num_kv_heads <= 0 || num_kv_heads > 65535 || num_heads % num_kv_heads) return -2;
  if (!(score_cap >= 0.f) || keep_first < 0 || weighting < 0 || weighting > 1 || (keep_first > 0 && window < 0)) return -2;
  if ((long)total_q * (num_heads / num_kv_heads) > 0x7fffffffL - 16) return -2;
  auto sixteen = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  if (!sixteen(q) || !sixteen(k_pages) || !sixteen(v_pages) || !sixteen(out) || q_stride % 4 || out_stride % 4) return -3;
  const FloatAttention p{q, k_pages, v_pages, out, block_tables, cu_seqlens_q, seq_lens_k, head_bias, ScoreTerms{score_cap, slopes, sinks},
                         q_stride, out_stride, bt_stride, num_seqs, num_heads, num_kv_heads, block_size, window, keep_first, weighting, scale};
  const int reach = window < 0 ? -window : window;
#define CASE(n)                                                                                             \
  case n:                                                                                                   \
    if (reach > 0 && reach <= kOneWaveWindow) return launch_float_attention<n, 1>(p, total_q, stream);      \
    if (reach > 0 && reach <= kTwoWaveWindow) return launch_float_attention<n, 2>(p, total_q, stream);      \
    return launch_float_attention<n, n <= 8 ? 8 : 4>(p, total_q, stream);
  switch (head_dim / 16) {
    CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8) CASE(9) CASE(10) CASE(11) CASE(12) CASE(13) CASE(14) CASE(15) CASE(16)
  }
#undef CASE
  return -2;
}
