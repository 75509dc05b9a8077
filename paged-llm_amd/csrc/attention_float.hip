// Paged causal attention of the true 32-bit path on the float matrix cores (v_mfma_f32_16x16x4_f32, exponentials and sums
// in float): head sizes that are multiples of 16 up to 256, pages whose size is a multiple of 16 positions.  The arrays,
// masks, score terms and weightings are those of attention_generic.hip, which keeps every other shape.
//
// A workgroup owns 16 columns, a column being a (query token, query head) pair of one sequence and one kv head, so that the
// heads of a group share every key and value that is loaded.  S^T = K Q^T leaves a lane with four keys of one column, which
// is the operand layout of O^T = V^T P^T as it stands: a lane's 16-byte load of V (four consecutive positions of a channel)
// meets its four weights in four instructions, and nothing is moved between lanes.
//
// The keys are cut into blocks of 32 (heads above 64: 16) at absolute positions.  Block b belongs to chain b mod 16, and a chain takes its blocks
// in ascending order with a running maximum of its own.  Chains g, g + 4, g + 8, g + 12 are joined in this order into group g, and the four
// groups in theirs.  That order is the same in both forms of the kernel, and a block that a column does not see changes none of
// its bits, so a column's result does not depend on how the tokens were cut into steps or batched.  Of a block that is seen in part,
// the tiles of 16 keys that no column sees are left out.
//   * One workgroup for a tile of columns: four wavefronts, a group each, its chains one after the other.
//   * Four workgroups, a group each, a wavefront a chain; what they leave is joined by a second kernel.  For few tiles (decoding).
// Which one is the host's choice (ops.float_attention_plan).
//
// What bounds it: the vector instructions of the softmax and the float instruction, half and half, where there are wavefronts enough, and a
// wavefront's chain of load, scores, exponentials and values where there are not.  So a block's keys are asked for before the softmax of the
// block in front of it and its values behind that block's, blocks are so small that keys, values and a group fit 168 registers (three
// wavefronts a SIMD; two for heads to 128, one beyond), and few tiles go to four times the compute units.  Against eight wavefronts a tile with
// blocks of 64 loaded as they come (32 heads of 64 on 4): decoding 8 requests at contexts to 700 18.5 -> 12.1 us, at 2,040 38 -> 18.3, one at 180 10.1 ->
// 8.0, 61 at contexts to 2,000 57 -> 46; prompts of 301 tokens 29.6 -> 17.5, 2,000 358 -> 266; 16 heads of 256 on one at 512 44 -> 19.3.  Over 576 shapes
// (1 to 61 sequences of 1 to 1,000 tokens at contexts of 60 to 3,000, heads of 64 to 256) 22 % less time with heads of 64, 27 % to 128 and 38 % beyond; what lies
// between the forms is slower: as many tiles as compute units with heads of 256 (200 tokens 23.7 -> 27.8, 1,000 172 -> 191), one head a kv head
// (16 requests at 700, 12 heads of 64: 21.9 -> 24.0), portions of 100 tokens behind 1,000 25.8 -> 26.3.
#include "common.h"

using namespace pllm;

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kColumns = 16, kTile = 16;

struct FloatAttention {
  const float *q, *k_pages, *v_pages;
  float* out;
  const int *block_tables, *cu_seqlens_q, *seq_lens_k;
  const float* head_bias;
  ScoreTerms terms;
  int q_stride, out_stride, bt_stride, num_seqs, num_heads, num_kv_heads, block_size, window, keep_first, weighting;
  float scale;
  float* parts;                                                        // (Z > 1) [groups][rows][D + 4]: a group's output, largest score and sum of weights
  int rows;                                                            // tokens x heads
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

// Lengths and page tables do not change while a launch runs: through the constant address space a load of them is a scalar load.
typedef const int __attribute__((address_space(4))) * ConstantInts;

// Where a chain of blocks stands: its largest score, the sum of its weights and its output so far.
template <int N> struct Standing { float m, l; f32x4 o[N]; };

// a and then b as one.
template <int N>
__device__ __forceinline__ void join(Standing<N>& a, const Standing<N>& b, bool softmax) {
  if (!softmax) {
#pragma unroll
    for (int t = 0; t < N; ++t) a.o[t] += b.o[t];
    return;
  }
  const float top = fmaxf(a.m, b.m), from = top == -INFINITY ? 0.f : top, fa = expf(a.m - from), fb = expf(b.m - from);
  a.m = top;
  a.l = fmaf(a.l, fa, b.l * fb);
#pragma unroll
  for (int t = 0; t < N; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j) a.o[t][j] = fmaf(a.o[t][j], fa, b.o[t][j] * fb);
}

// All of a column's groups, and the division by the sum of weights.  (A group without a key adds nothing: its largest score is -inf.)
template <int GROUPS>
__device__ __forceinline__ f32x4 join_groups(const Standing<1> (&g)[GROUPS], bool softmax) {
  float top = g[0].m, sum = 0.f;
#pragma unroll
  for (int w = 1; w < GROUPS; ++w) top = fmaxf(top, g[w].m);
  f32x4 out{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int w = 0; w < GROUPS; ++w) {
    const float factor = softmax ? expf(g[w].m - top) : 1.f;           // (top is finite: a query sees itself)
    sum = fmaf(g[w].l, factor, sum);
#pragma unroll
    for (int j = 0; j < 4; ++j) out[j] = fmaf(g[w].o[0][j], factor, out[j]);
  }
  return softmax ? out * (1.f / sum) : out;
}

// DT: head size / 16.  KEYS: of a block.  GROUPS, SUBS: the groups and the chains of one (above: 4 and 4; layers of short windows have fewer).
// Z: workgroups of a tile of columns; with more than one another kernel joins the groups.
template <int DT, int KEYS, int WAVES, int GROUPS, int SUBS, int PER_SIMD, int Z>
__global__ __launch_bounds__(64 * WAVES, PER_SIMD) void paged_attention_float_kernel(FloatAttention p) {
  constexpr int D = 16 * DT, kChunk = DT < 8 ? DT : 8, kBlock = KEYS, kTiles = KEYS / kTile, kChains = GROUPS * SUBS;
  constexpr bool kEarly = DT <= 4 || KEYS < 64;                        // registers for a whole block's keys and values at once
  constexpr int kGroups = GROUPS / Z, kSharing = WAVES / kGroups, kEach = SUBS / kSharing;   // a workgroup's groups, wavefronts of one, chains of one
  static_assert(GROUPS % Z == 0 && WAVES % kGroups == 0 && SUBS % kSharing == 0, "equal shares");
  constexpr int kSlots = kSharing == 1 ? WAVES : kGroups * SUBS;       // a group that one wavefront has, or a chain
  __shared__ float lds_m[kSlots][kColumns], lds_l[kSlots][kColumns];
  __shared__ int lds_live[kSlots];                                     // whether a block has been seen
  extern __shared__ __attribute__((aligned(16))) unsigned char fa_lds[];
  f32x4* lds_o = reinterpret_cast<f32x4*>(fa_lds);                     // [kSlots][DT][64]
  const int tid = threadIdx.x, lane = tid & 63, column = lane & 15, quad = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = p.num_heads / p.num_kv_heads, kvh = blockIdx.y;

  // Sequence s has the tiles from floor(cu[s] group / 16) + s on; those that its columns do not fill end at once.  With one token a
  // sequence the tile's sequence follows from its number, which is looked at first: one trip to memory in place of one a halving.
  ConstantInts cu = (ConstantInts)p.cu_seqlens_q, lens = (ConstantInts)p.seq_lens_k;
  auto tiles_before = [&](int s, int tokens) { return (int)((long)tokens * group / kColumns) + s; };
  int seq = min((int)(((long)blockIdx.x * kColumns + kColumns - 1) / (kColumns + group)), p.num_seqs - 1);
  int q_begin = cu[seq], q_end = cu[seq + 1], len_k = lens[seq];
  if (tiles_before(seq, q_begin) > (int)blockIdx.x || (seq + 1 < p.num_seqs && tiles_before(seq + 1, q_end) <= (int)blockIdx.x)) {
    int lo = 0, hi = p.num_seqs - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (tiles_before(mid, cu[mid]) <= (int)blockIdx.x) lo = mid; else hi = mid - 1;
    }
    seq = lo;
    q_begin = cu[seq], q_end = cu[seq + 1], len_k = lens[seq];
  }
  const int num_q = q_end - q_begin;
  const int first_column = ((int)blockIdx.x - ((int)((long)q_begin * group / kColumns) + seq)) * kColumns;
  const long columns = (long)num_q * group;
  if (first_column >= columns) return;
  ConstantInts bt = (ConstantInts)p.block_tables + (size_t)seq * p.bt_stride;
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
  // (a page of one tile, the usual size, needs no division)
  const int page_tiles = p.block_size / kTile;
  auto page_at = [&](int n) { return page_tiles == 1 ? n / kTile : n / kTile / page_tiles; };
  auto inside = [&](int n) { return page_tiles == 1 ? n % kTile : n % p.block_size; };
  const int page_last = bt[page_at(pos_max)];
  // The blocks that this wavefront visits, chain after chain: (sub, b), sub past the last chain at the end.
  const int own_group = wave % kGroups, first_sub = wave / kGroups * kEach;
  auto chain_of = [&](int sub) { return (int)blockIdx.z * kGroups + own_group + (first_sub + sub) * GROUPS; };
  auto settle = [&](int& sub, int& b) {
    while (sub < kEach) {
      if (b * kBlock > pos_max) {
        b = chain_of(++sub);
      } else if (b * kBlock + kBlock - 1 < any_from && b * kBlock >= p.keep_first) {   // between the kept positions and the window: on to its first
        b += (any_from / kBlock - b + kChains - 1) / kChains * kChains;
      } else {
        return;
      }
    }
  };
  int page_of[kTiles];
  auto ask_pages = [&](int b) {
#pragma unroll
    for (int i = 0; i < kTiles; ++i) page_of[i] = bt[page_at(min(b * kBlock + i * kTile, pos_max))];
  };
  const int lane_k = column * D + 4 * quad, lane_v = column * p.block_size + 4 * quad;   // a lane's place in a tile
  struct Place {                                                       // a tile lies inside one page: the first elements of its keys and values
    const float *k[kTiles], *v[kTiles];
    bool live[kTiles], all_live;                                       // (the same for all lanes: a tile that no column sees is left out)
  };
  auto place_of = [&](int b) {
    Place at;
    at.all_live = true;
#pragma unroll
    for (int i = 0; i < kTiles; ++i) {
      const int n = b * kBlock + i * kTile;
      at.live[i] = n <= pos_max && (n + kTile > any_from || n < p.keep_first);
      at.all_live = at.all_live && at.live[i];
      const int from = at.live[i] ? n : pos_max / kTile * kTile;       // (a tile that no column sees: any valid one, for loads without conditions)
      const size_t page = (size_t)(at.live[i] ? page_of[i] : page_last) * p.num_kv_heads + kvh;
      at.k[i] = p.k_pages + (page * p.block_size + inside(from)) * D;
      at.v[i] = p.v_pages + page * D * p.block_size + inside(from);
    }
    return at;
  };
  // A block's keys are asked for behind the scores of the block before it, its values behind that block's values.
  f32x4 k_early[kEarly ? kTiles : 1][kEarly ? DT : 1], v_early[kEarly ? kTiles : 1][kEarly ? DT : 1];
  auto ask_keys = [&](const Place& at) {
#pragma unroll
    for (int i = 0; i < (kEarly ? kTiles : 0); ++i)
#pragma unroll
      for (int t = 0; t < DT; ++t) k_early[kEarly ? i : 0][kEarly ? t : 0] = *reinterpret_cast<const f32x4*>(at.k[i] + 16 * t + lane_k);
  };
  auto ask_values = [&](const Place& at) {
#pragma unroll
    for (int i = 0; i < (kEarly ? kTiles : 0); ++i)
#pragma unroll
      for (int t = 0; t < DT; ++t) v_early[kEarly ? i : 0][kEarly ? t : 0] = *reinterpret_cast<const f32x4*>(at.v[i] + (size_t)16 * t * p.block_size + lane_v);
  };

  Standing<DT> group_so_far, now;                                      // the chains before joined in order (where a wavefront has several), and this one
  float &m = now.m, &l = now.l;                                        // (l: this lane's share of the column's sum until the chain's end)
  auto& o = now.o;
  bool group_live = false, chain_live = false;
  auto begin_chain = [&]() {
    m = -INFINITY;
    l = 0.f;
#pragma unroll
    for (int t = 0; t < DT; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    chain_live = false;
  };
  auto hand_over = [&](int slot, const Standing<DT>& what) {
    if (quad == 0) {
      lds_m[slot][column] = what.m;
      lds_l[slot][column] = what.l;
    }
    if (lane == 0) lds_live[slot] = 1;
#pragma unroll
    for (int t = 0; t < DT; ++t) lds_o[(slot * DT + t) * 64 + lane] = what.o[t];
  };
  if (tid < kSlots) lds_live[tid] = 0;
  __syncthreads();
  auto end_chain = [&](int sub) {
    if (!chain_live) return;
    l = column_sum(l);
    if (kSharing > 1) {
      hand_over(own_group * SUBS + first_sub + sub, now);
    } else {
      if (kEach > 1 && group_live) join(group_so_far, now, softmax); else group_so_far = now;
      group_live = true;
    }
  };
  begin_chain();
  if (p.terms.sinks && softmax && chain_of(0) == 0) {                  // as if one key with this score and no value had been seen
    m = p.terms.sinks[head];
    l = quad == 0 ? 1.f : 0.f;
    chain_live = true;
  }
  int sub = 0, b = chain_of(0);
  settle(sub, b);
  if (sub > 0) {
    end_chain(0);
    begin_chain();
  }
  Place at;
  if (sub < kEach) {
    ask_pages(b);
    at = place_of(b);
    ask_keys(at);
    ask_values(at);
  }
#pragma unroll 1
  while (sub < kEach) {
    const int n0 = b * kBlock;
    int next_sub = sub, next_b = b + kChains;
    settle(next_sub, next_b);
    const bool more = next_sub < kEach;
    ask_pages(more ? next_b : b);
    chain_live = true;
    const bool whole = n0 + kBlock - 1 <= pos_min && n0 >= all_from;   // every column sees every key of the block
    f32x4 s[kTiles];
#pragma unroll
    for (int i = 0; i < kTiles; ++i) s[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (kEarly && at.all_live) {
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int i = 0; i < kTiles; ++i) s[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(k_early[kEarly ? i : 0][kEarly ? t : 0][j], q[t][j], s[i], 0, 0, 0);
    } else {
#pragma unroll
      for (int i = 0; i < kTiles; ++i) {
        if (!at.live[i]) continue;
#pragma unroll
        for (int t0 = 0; t0 < DT; t0 += kChunk) {
          f32x4 k[kChunk];
#pragma unroll
          for (int t = 0; t < kChunk; ++t)
            if (t0 + t < DT) k[t] = kEarly ? k_early[kEarly ? i : 0][kEarly ? t0 + t : 0] : *reinterpret_cast<const f32x4*>(at.k[i] + 16 * (t0 + t) + lane_k);
#pragma unroll
          for (int t = 0; t < kChunk; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j)
              if (t0 + t < DT) s[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[t][j], q[t0 + t][j], s[i], 0, 0, 0);
        }
      }
    }
    const Place next = place_of(more ? next_b : b);
    if (more) ask_keys(next);
    auto seen = [&](int n) { return whole || (n <= pos && (n >= first_key || n < p.keep_first)); };
    auto each_score = [&](auto change) {
#pragma unroll
      for (int i = 0; i < kTiles; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) s[i][j] = change(s[i][j], n0 + i * kTile + 4 * quad + j);
    };
    each_score([&](float x, int) { return x * p.scale; });
    if (p.terms.cap > 0.f) each_score([&](float x, int) { return capped_score(x, p.terms.cap); });
    if (p.terms.slopes) each_score([&](float x, int n) { return x + slope * (float)(n - pos); });
    if (softmax) {
      if (!whole) each_score([&](float x, int n) { return seen(n) ? x : -INFINITY; });
      float top = m;
#pragma unroll
      for (int i = 0; i < kTiles; ++i) top = fmaxf(top, fmaxf(fmaxf(s[i][0], s[i][1]), fmaxf(s[i][2], s[i][3])));
      top = column_max(top);
      const float from = top == -INFINITY ? 0.f : top;                 // (a column that has seen no key yet)
      const float alpha = expf(m - from);
      float sum = 0.f;
      each_score([&](float x, int) {
        const float weight = expf(x - from);
        sum += weight;
        return weight;
      });
      m = top;
      l = l * alpha + sum;
      if (__any(alpha != 1.f)) {
#pragma unroll
        for (int t = 0; t < DT; ++t) o[t] *= alpha;
      }
    } else {
      each_score([&](float x, int n) { return seen(n) ? 1.f / (1.f + expf(-(x + bias))) : 0.f; });
    }
#pragma unroll
    for (int i = 0; i < kTiles; ++i) {
      if (!at.live[i]) continue;
#pragma unroll
      for (int t0 = 0; t0 < DT; t0 += kChunk) {
        const int n = n0 + i * kTile;
        f32x4 own_v[kEarly ? 1 : kChunk];
        f32x4* v = kEarly ? v_early[kEarly ? i : 0] + t0 : own_v;
        if (!kEarly) {
#pragma unroll
          for (int t = 0; t < kChunk; ++t)
            if (t0 + t < DT) v[t] = *reinterpret_cast<const f32x4*>(at.v[i] + (size_t)16 * (t0 + t) * p.block_size + lane_v);
        }
        if (!whole) {
          // A weight of zero must not meet a value that is no number.  Where there is one among the tile's: slots that no column
          // sees hold anything (zeros instead), and a value that is not finite is left out here and given to the columns that see it,
          // one by one.
          float zero = 0.f;                                            // (or NaN)
#pragma unroll
          for (int t = 0; t < kChunk; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j)
              if (t0 + t < DT) zero = fmaf(v[t][j], 0.f, zero);
          if (__any(!(zero == 0.f))) {
#pragma unroll
            for (int t = 0; t < kChunk; ++t)
#pragma unroll
              for (int j = 0; j < 4; ++j)
                if (t0 + t < DT) v[t][j] = fabsf(v[t][j]) < INFINITY ? v[t][j] : 0.f;
#pragma unroll 1
            for (int key = 0; key < kTile; ++key) {
              const float own = key % 4 == 0 ? s[i][0] : key % 4 == 1 ? s[i][1] : key % 4 == 2 ? s[i][2] : s[i][3];
              const float weight = __shfl(own, (key / 4) * 16 + column);
              if (n + key > pos_max || !seen(n + key)) continue;
              int from = 4 * quad * p.block_size + key;                // (its address is formed anew for every key: this path is rare and has no
              asm volatile("" : "+v"(from));                           //  registers to spare)
#pragma unroll
              for (int t = 0; t < kChunk; ++t) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                  if (t0 + t < DT) {
                    const float x = at.v[i][from + (16 * (t0 + t) + j) * p.block_size];
                    if (!(fabsf(x) < INFINITY)) o[t0 + t][j] = fmaf(weight, x, o[t0 + t][j]);
                  }
                __builtin_amdgcn_sched_barrier(0);
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
    if (more) ask_values(next);
    if (next_sub > sub) {
      end_chain(sub);
      begin_chain();
    }
    sub = next_sub;
    b = next_b;
    at = next;
  }

  if (kSharing == 1 && group_live) hand_over(wave, group_so_far);
  __syncthreads();
  if (first_column + column > last_column) return;
  // One of the workgroup's groups, its chains in their order, of 16 channels.
  auto group_of = [&](int w, int t) {
    constexpr int kParts = kSharing == 1 ? 1 : SUBS;
    Standing<1> g{-INFINITY, 0.f, {f32x4{0.f, 0.f, 0.f, 0.f}}};
    bool live = false;
#pragma unroll
    for (int i = 0; i < kParts; ++i) {
      const int slot = w * kParts + i;
      if (!__builtin_amdgcn_readfirstlane(lds_live[slot])) continue;
      const Standing<1> part{lds_m[slot][column], lds_l[slot][column], {lds_o[(slot * DT + t) * 64 + lane]}};
      if (live) join(g, part, softmax); else g = part;
      live = true;
    }
    return g;
  };
  for (int t = wave; t < DT; t += WAVES) {                             // (the groups' largest scores and sums are those of every t)
    Standing<1> g[kGroups];
#pragma unroll
    for (int w = 0; w < kGroups; ++w) g[w] = group_of(w, t);
    if constexpr (Z == 1) {
      *reinterpret_cast<f32x4*>(p.out + (size_t)tok * p.out_stride + (size_t)head * D + 16 * t + 4 * quad) = join_groups<GROUPS>(g, softmax);
    } else {
#pragma unroll
      for (int w = 0; w < kGroups; ++w) {
        float* part = p.parts + ((size_t)(blockIdx.z * kGroups + w) * p.rows + (size_t)tok * p.num_heads + head) * (D + 4);
        *reinterpret_cast<f32x4*>(part + 16 * t + 4 * quad) = g[w].o[0];
        if (t == 0 && quad == 0) *reinterpret_cast<f32x2*>(part + D) = f32x2{g[w].m, g[w].l};
      }
    }
  }
}

// The groups that several workgroups have, joined: a thread has four channels of a row.
template <int GROUPS>
__global__ __launch_bounds__(256) void join_float_parts_kernel(FloatAttention p, int D) {
  const int each = D / 4, at = blockIdx.x * 256 + threadIdx.x, row = at / each, c = 4 * (at - row * each);
  if (row >= p.rows) return;
  Standing<1> g[GROUPS];
#pragma unroll
  for (int w = 0; w < GROUPS; ++w) {
    const float* part = p.parts + ((size_t)w * p.rows + row) * (D + 4);
    const f32x2 ml = *reinterpret_cast<const f32x2*>(part + D);
    g[w] = Standing<1>{ml[0], ml[1], {*reinterpret_cast<const f32x4*>(part + c)}};
  }
  const int tok = row / p.num_heads, head = row - tok * p.num_heads;
  *reinterpret_cast<f32x4*>(p.out + (size_t)tok * p.out_stride + (size_t)head * D + c) = join_groups<GROUPS>(g, p.weighting == 0);
}

// One or two wavefronts, a chain of blocks of 64 keys each, for layers whose window is so short that a tile of columns sees keys of two to four
// such blocks only.  Further wavefronts would find no block, and keep other workgroups off the compute unit (200 requests at context
// 300, 16 heads of 64: a window of 30 29 us with one wavefront and 69 with four, a window of 100 53 us with two and 78 with four).  The window is the
// layer's, so a layer's columns keep their order of additions in every step.  (Relative error against 64 bits / in the plain kernel, 700
// positions: window 30 3.29e-7 / 3.27e-7, 100 4.38e-7 / 4.50e-7; one wavefront at 64 would have 4.10e-7 against 4.03e-7.)
constexpr int kOneWaveWindow = 32, kTwoWaveWindow = 128;

template <int DT, int KEYS, int WAVES, int GROUPS, int SUBS, int PER_SIMD, int Z>
static int launch_float_attention(const FloatAttention& p, int total_q, hipStream_t stream) {
  const int group = p.num_heads / p.num_kv_heads;
  const dim3 grid((unsigned)((long)total_q * group / kColumns + p.num_seqs), p.num_kv_heads, Z), block(64 * WAVES);
  const size_t lds = (size_t)WAVES * DT * 64 * sizeof(f32x4);
  auto kernel = paged_attention_float_kernel<DT, KEYS, WAVES, GROUPS, SUBS, PER_SIMD, Z>;
  if (lds > 48 * 1024) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return (int)e;
  }
  hipLaunchKernelGGL(kernel, grid, block, lds, stream, p);
  if (Z > 1) {
    const long threads = (long)p.rows * (DT * 4);
    hipLaunchKernelGGL(join_float_parts_kernel<GROUPS>, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream, p, 16 * DT);
  }
  PLLM_RETURN_LAST_ERROR();
}

// cut: workgroups of a tile of columns, 1 or 4; beyond one, `parts` [4][total_q * num_heads][head_dim + 4] floats on a 16-byte boundary.  Windows
// up to kTwoWaveWindow have one workgroup whatever `cut` says.
PLLM_API int pllm_paged_attention_float(const float* q, int q_stride, const float* k_pages, const float* v_pages, float* out, int out_stride,
                                        const int* block_tables, int bt_stride, const int* cu_seqlens_q, const int* seq_lens_k, int num_seqs,
                                        int total_q, int num_heads, int num_kv_heads, int head_dim, int block_size, float scale, int window,
                                        float score_cap, const float* slopes, const float* sinks, int keep_first, int weighting,
                                        const float* head_bias, int cut, float* parts, hipStream_t stream) {
  if (total_q <= 0 || num_seqs <= 0) return 0;
  if (head_dim <= 0 || head_dim % 16 || head_dim > 256 || block_size <= 0 || block_size % kTile) return -2;
  if (num_kv_heads <= 0 || num_kv_heads > 65535 || num_heads % num_kv_heads) return -2;
  if (!(score_cap >= 0.f) || keep_first < 0 || weighting < 0 || weighting > 1 || (keep_first > 0 && window < 0)) return -2;
  if ((long)total_q * (num_heads / num_kv_heads) > 0x7fffffffL - 16) return -2;
  auto sixteen = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  if (!sixteen(q) || !sixteen(k_pages) || !sixteen(v_pages) || !sixteen(out) || q_stride % 4 || out_stride % 4) return -3;
  const FloatAttention p{q, k_pages, v_pages, out, block_tables, cu_seqlens_q, seq_lens_k, head_bias, ScoreTerms{score_cap, slopes, sinks},
                         q_stride, out_stride, bt_stride, num_seqs, num_heads, num_kv_heads, block_size, window, keep_first, weighting, scale, parts, total_q * num_heads};
  const int reach = window < 0 ? -window : window;
  if (cut != 1 && (cut != 4 || !parts || !sixteen(parts))) return -2;
#define CASE(n)                                                                                             \
  case n:                                                                                                   \
    if (reach > 0 && reach <= kOneWaveWindow) return launch_float_attention<n, 64, 1, 1, 1, n <= 8 ? 2 : 1, 1>(p, total_q, stream);   \
    if (reach > 0 && reach <= kTwoWaveWindow) return launch_float_attention<n, 64, 2, 2, 1, n <= 8 ? 2 : 1, 1>(p, total_q, stream);   \
    if (cut == 4) return launch_float_attention<n, n <= 4 ? 32 : 16, 4, 4, 4, n <= 4 ? 3 : n <= 8 ? 2 : 1, 4>(p, total_q, stream);    \
    return launch_float_attention<n, n <= 4 ? 32 : 16, 4, 4, 4, n <= 4 ? 3 : n <= 8 ? 2 : 1, 1>(p, total_q, stream);
  switch (head_dim / 16) {
    CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8) CASE(9) CASE(10) CASE(11) CASE(12) CASE(13) CASE(14) CASE(15) CASE(16)
  }
#undef CASE
  return -2;
}
