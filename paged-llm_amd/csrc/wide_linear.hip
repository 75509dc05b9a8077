// Products of prompt steps: y = x W^T for bfloat16 rows and a tiled weight matrix (ops.tile_weight), in tiles of 64 x 64 to 128 x 160
// outputs, one workgroup of four wavefronts a tile, with bfloat16 or float results, act(gate) * up, or the rotation of q and k
// with the write of k and v into their cache pages behind; gated products, and plain ones in fewer rounds than the library has, in tiles of up to 320 x 256
// and 256 x 352 by eight wavefronts (big_linear_kernel).
//
// What bounds it: the matrix cores at the clock that they hold under such a load (1.3 to 1.4 PFLOP/s over the chip with nothing else in the
// kernel), and for tiles of 128 x 128 and less a compute unit's way to the L2 (26 to 45 bytes a clock).  So every other
// instruction has to hide behind the products, and one wavefront per SIMD with up to 512 registers does that:
//   * Stages of 64 columns lie in LDS, R of them, filled by global_load_lds (16 bytes a lane, no registers in between): weights in whole
//     kilobytes in operand order, rows in pieces of 128 bytes in an order that spreads the banks.
//   * A stage's columns are two steps of 32.  While the products of one step run, the operands of the next come from LDS; in the middle of
//     a stage, behind the only barrier, its slot is free and the loads of the stage R ahead are issued.
//   * Loads, LDS reads and products are dealt out evenly in the source and kept there: the loads of a stage in front of its
//     products hold up the wavefront until the memory pipe has taken them all.
//   * The sums are held in the accumulation registers by the instruction's own operand constraint: left to itself the compiler moves
//     them to and fro (96 to 248 moves a stage).
// Measured (us, weights from memory; in brackets the library's product, with the kernel behind it where there is one): 896 rows x 2048 x 2048 14.0 (16.4),
// 512 x 1024 x 1024 5.7 (8.4), 2048 x 2048 x 4096 39.5 (40.4), gated 512 rows of 5632 x 1024 13.4 (20.6), 320 rows of 11264 x 2048 25.4 (33.0).
// Which tile a product takes, and whether it comes here, is the host's choice (ops.wide_linear_plan, ops.wide_gated_plan, ops.wide_plain_plan, ops.wide_rotary_plan).
// An output is one chain in ascending k whatever its tile.
// moe_wide.hip has the same stages, waits and held sums for the experts' products: what is mended in one belongs in the other.
#include "common.h"
#include <type_traits>

using namespace pllm;

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float floatx4;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

enum { WL_BF16 = 0, WL_F32 = 1, WL_GATED = 2, WL_ROPE_KV = 4 };

struct WideParams {
  const bf16* x;
  const bf16* wt;             // [blocks of 16 rows][K / 32][64 lanes][8]
  void* out;
  int ldx, ldo, M, N, ksteps, weight_blocks, n_blocks, m_blocks;        // N: outputs (gated: half the weight rows)
  int activation, num_heads, num_kv_heads, head_dim, block_size;
  const int *positions, *slots;
  const float *cos_t, *sin_t;
  bf16 *k_pages, *v_pages;
};

template <int N_>
__device__ __forceinline__ void wait_loads_but() {   // until at most N_ of this wavefront's loads are still under way
  static_assert(N_ >= 0 && N_ < 64, "vmcnt has six bits");
  __builtin_amdgcn_s_waitcnt((N_ & 0xf) | ((N_ >> 4) << 14) | 0x0f70);
}

// The larger of m and two magnitudes; NaN counts as nothing.
__device__ __forceinline__ float largest(float a, float b, float m) {
  float o;
  asm("v_max3_f32 %0, |%1|, |%2|, %3" : "=v"(o) : "v"(a), "v"(b), "v"(m));
  return o;
}

// act(z) of COUNT values as z / (1 + exp(-v)), v = z for SiLU and 2 sqrt(2 / pi) (z + 0.044715 z^3) for GELU in its form with tanh: the quotient's first value
// corrected once, which leaves the error that expf and a division have (SiLU relative to 64 bits, z from -87 to 87: RMS 3.6e-8, at most 1.8e-7) at half of
// their instructions, without a branch inside.  False where some results are to be made another way: magnitudes from quick_limit on (NaN is right as it is).
__device__ __forceinline__ float quick_limit(int act) { return act == PLLM_ACT_SILU ? 87.f : 3e38f; }

template <int COUNT>
__device__ __forceinline__ bool quick_gate(const float (&z)[COUNT], float (&out)[COUNT], int act) {
#pragma clang fp contract(off)
  static_assert(COUNT % 2 == 0, "pairs");
  // exp(-v) from the instruction for 2^x: -v / ln 2 as a rounded product and what the rounding left, the whole part put into the exponent.  In three passes,
  // so that no instruction waits for the slow one in front of it.
  float most = 0.f, e[COUNT], part[COUNT];
  int whole[COUNT];
  if (act == PLLM_ACT_SILU) {
#pragma unroll
    for (int i = 0; i < COUNT; ++i) e[i] = z[i];
  } else {
#pragma unroll
    for (int i = 0; i < COUNT; ++i) e[i] = __builtin_amdgcn_fmed3f(z[i] * fmaf(z[i] * z[i], 0.0713548163f, 1.59576912f), -87.f, 87.f);
  }
#pragma unroll
  for (int i = 0; i < COUNT; ++i) {
    const float v = -e[i], t = v * 1.44269504f, n = __builtin_rintf(t);
    e[i] = __builtin_amdgcn_exp2f((t - n) + fmaf(v, 1.9259629911e-8f, fmaf(v, 1.44269504f, -t)));
    whole[i] = (int)n;
    if (i & 1) most = largest(z[i - 1], z[i], most);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < COUNT; ++i) {
    e[i] = 1.f + __builtin_ldexpf(e[i], whole[i]);
    part[i] = __builtin_amdgcn_rcpf(e[i]);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < COUNT; ++i) {
    const float q = z[i] * part[i];
    out[i] = fmaf(fmaf(-q, e[i], z[i]), part[i], q);
  }
  return __all(most < quick_limit(act));
}

// act(z) times y in place of z, for the results of a lane that lie in one row.
template <int COUNT>
__device__ __forceinline__ void gate(float (&z)[COUNT], const float (&y)[COUNT], int act) {
  float quick[COUNT];
  if (!quick_gate(z, quick, act)) {
#pragma unroll
    for (int i = 0; i < COUNT; ++i)
      if (!(fabsf(z[i]) < quick_limit(act))) quick[i] = gate_activation(z[i], act);
  }
#pragma unroll
  for (int i = 0; i < COUNT; ++i) z[i] = quick[i] * y[i];
}

// Products that take two weight rows: rows 8-15 of a block (the lanes 32 further on) are the partners of rows 0-7.  The halves change places so
// that lanes 0-31 have rows 4 g, 4 g + 1 and lanes 32-63 rows 4 g + 2, 4 g + 3, with their partners: from row (g & 1) * 4 + (g >> 1) * 2 on.
__device__ __forceinline__ void swap_halves(const floatx4& a, float* one, float* other) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(a[i]), __float_as_uint(a[i + 2]), false, false);
    one[i] = __uint_as_float(x[0]);
    other[i] = __uint_as_float(x[1]);
  }
}

__device__ __forceinline__ unsigned two_bf16(float x, float y) {
  return __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{x, y}, bf16x2));
}

// What is done with a wavefront's sums: MW tiles of 16 rows from row0 on x NW blocks of 16 weight rows from block unit0 on.
template <int EPI, int MW, int NW>
__device__ __forceinline__ void finish(const WideParams& p, const floatx4 (&acc)[MW][NW], int row0, int unit0, int lane) {
  const int r = lane & 15, g = lane >> 4;
  // A lane's four sums are four weight rows (4 g .. 4 g + 3 of the block) of input row r of the tile.  Stores go through a buffer that drops what
  // lies past its end, so that no store has a branch of its own (with branches the end of 128 x 128 took 3 us longer).
  const int row_bytes = p.ldo * (EPI == WL_F32 ? 4 : 2);
  const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(p.out, 0, (int)((unsigned)p.M * (unsigned)row_bytes), 0x00027000);
  const int pair_row = (g & 1) * 4 + (g >> 1) * 2;                     // (of swap_halves)
  // A rotation's operands are asked for together: one by one each waits for the memory, and for the stores in front of it (2048 rows of 2560 x 2048
  // 35.2 -> 33 us, 777 of 3072 x 2048 23.7 -> 20.3, 26.7 and 16 without the rotation; the tiled kernel, with two blocks on a compute unit, gains nothing).
  constexpr bool kTurns = EPI == WL_ROPE_KV;
  int pos[kTurns ? MW : 1], slots[kTurns ? MW : 1];
  f32x2 turn[kTurns ? MW : 1][kTurns ? NW : 1][2];
  int heads[kTurns ? NW : 1], rows_in[kTurns ? NW : 1];                // a block's head, and this lane's first row in the head's half
  if constexpr (kTurns) {
#pragma unroll
    for (int t = 0; t < MW; ++t) {
      const int m = min(row0 + t * 16 + r, p.M - 1);
      pos[t] = p.positions[m];
      slots[t] = p.slots[m];
    }
    const int half = p.head_dim >> 1, per_head = half >> 3;
    int head = unit0 / per_head, in_head = unit0 - head * per_head;
#pragma unroll
    for (int u = 0; u < NW; ++u) {
      heads[u] = head;
      rows_in[u] = in_head * 8 + pair_row;
      if (++in_head == per_head) in_head = 0, ++head;
    }
#pragma unroll
    for (int t = 0; t < MW; ++t)
#pragma unroll
      for (int u = 0; u < NW; ++u) {
        const size_t at = (size_t)pos[t] * half + rows_in[u];
        turn[t][u][0] = p.cos_t ? *reinterpret_cast<const f32x2*>(p.cos_t + at) : f32x2{1.f, 1.f};
        turn[t][u][1] = p.cos_t ? *reinterpret_cast<const f32x2*>(p.sin_t + at) : f32x2{0.f, 0.f};
      }
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int t = 0; t < MW; ++t) {
    const int m = row0 + t * 16 + r;
    const int at_row = m * row_bytes;
    if constexpr (EPI == WL_GATED) {
      float z[2 * NW], y[2 * NW];
#pragma unroll
      for (int u = 0; u < NW; ++u) swap_halves(acc[t][u], z + 2 * u, y + 2 * u);
      gate(z, y, p.activation);
#pragma unroll
      for (int u = 0; u < NW; ++u) {
        const int c = (unit0 + u) * 8 + pair_row;
        __builtin_amdgcn_raw_buffer_store_b32(two_bf16(z[2 * u], z[2 * u + 1]), out, c < p.N && m < p.M ? at_row + 2 * c : -1, 0, 0);
      }
      continue;
    }
    const int slot_kv = kTurns && m < p.M ? slots[kTurns ? t : 0] : -1;
    int page = 0, off = 0;
    if (kTurns && heads[kTurns ? NW - 1 : 0] >= p.num_heads && slot_kv >= 0) page = slot_kv / p.block_size, off = slot_kv - page * p.block_size;
#pragma unroll
    for (int u = 0; u < NW; ++u) {
      const floatx4 a = acc[t][u];
      const int unit = unit0 + u;
      if constexpr (EPI == WL_F32) {
        const int c = unit * 16 + g * 4;
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, a), out, c < p.N && m < p.M ? at_row + 4 * c : -1, 0, 0);
      } else if constexpr (EPI == WL_BF16) {
        const int c = unit * 16 + g * 4;
        __builtin_amdgcn_raw_buffer_store_b64(u32x2{two_bf16(a[0], a[1]), two_bf16(a[2], a[3])}, out, c < p.N && m < p.M ? at_row + 2 * c : -1, 0, 0);
      } else {
        float x[2], y[2];
        swap_halves(a, x, y);
        const int d = p.head_dim, half = d >> 1, nh = p.num_heads, nkv = p.num_kv_heads, head = heads[u], ri = rows_in[u];
        if (head >= nh + 2 * nkv) continue;
        if (head < nh + nkv) {
          const f32x2 cs = turn[t][u][0], sn = turn[t][u][1];
          float lo[2], hi[2];
#pragma unroll
          for (int i = 0; i < 2; ++i)
            rotate_pair(__bfloat162float(__float2bfloat16(x[i])), __bfloat162float(__float2bfloat16(y[i])), cs[i], sn[i], lo[i], hi[i]);
          if (head < nh) {
            const int at = m < p.M ? at_row + 2 * (head * d + ri) : -1;
            __builtin_amdgcn_raw_buffer_store_b32(two_bf16(lo[0], lo[1]), out, at, 0, 0);
            __builtin_amdgcn_raw_buffer_store_b32(two_bf16(hi[0], hi[1]), out, m < p.M ? at + 2 * half : -1, 0, 0);
          } else if (slot_kv >= 0) {
            bf16* dst = p.k_pages + (((size_t)page * nkv + (head - nh)) * p.block_size + off) * d + ri;
            *reinterpret_cast<unsigned*>(dst) = two_bf16(lo[0], lo[1]);
            *reinterpret_cast<unsigned*>(dst + half) = two_bf16(hi[0], hi[1]);
          }
        } else if (slot_kv >= 0) {                                   // values stand transposed in their page; 16 tokens in a row fill a row of it
          bf16* dst = p.v_pages + (((size_t)page * nkv + (head - nh - nkv)) * d + ri) * p.block_size + off;
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            dst[(size_t)i * p.block_size] = __float2bfloat16(x[i]);
            dst[(size_t)(half + i) * p.block_size] = __float2bfloat16(y[i]);
          }
        }
      }
    }
  }
}

// Wavefronts WM x 4 / WM, each with MW tiles of 16 rows x NW blocks of 16 weight rows.
template <int EPI, int WM, int MW, int NW, int R>
__global__ __launch_bounds__(256, 1) void wide_linear_kernel(WideParams p) {
  constexpr int WN = 4 / WM, NB = WN * NW, XT = WM * MW;               // blocks of weight rows, tiles of rows of the workgroup
  constexpr int kSlot = (NB + XT) * 2048;                              // bytes of a stage: two steps of every block and tile
  constexpr int LW = (NB * 2 + 3) / 4, LX = (XT * 2 + 3) / 4, L = LW + LX, F = MW + NW;   // a wavefront's loads of a stage, its operands of a step
  constexpr int Q = L > F ? L : F;                                     // shares that a step is dealt out in
  extern __shared__ __attribute__((aligned(16))) unsigned char wl_lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // The blocks of rows of one tile of weight rows follow each other on one XCD (workgroup b runs on XCD b % 8); the last group
  // has fewer than eight tiles of weight rows where their number is no multiple of 8.
  const int group = blockIdx.x / (8 * p.m_blocks), in_group = blockIdx.x - group * 8 * p.m_blocks, across = min(8, p.n_blocks - group * 8);
  const int nb = group * 8 + in_group % across, row0 = in_group / across * (XT * 16);
  const int n = p.ksteps >> 1;                                         // stages

  const bf16 *wbase[LW], *xbase[LX];                                   // (a share that is one load short repeats its last one)
#pragma unroll
  for (int i = 0; i < LW; ++i) {
    const int bb = min(wave + 4 * i, NB * 2 - 1);
    wbase[i] = p.wt + (((size_t)min(nb * NB + (bb >> 1), p.weight_blocks - 1) * p.ksteps + (bb & 1)) * 64 + lane) * 8;
  }
  const int xr = lane >> 3, xg = (lane & 7) ^ xr;                      // a load: 8 rows x 128 bytes, the row's pieces in XOR-ed order
#pragma unroll
  for (int i = 0; i < LX; ++i) {
    const int bb = min(wave + 4 * i, XT * 2 - 1);
    xbase[i] = p.x + (size_t)min(row0 + bb * 8 + xr, p.M - 1) * p.ldx + xg * 8;             // rows past the end repeat the last one
  }
  auto issue = [&](int i, int s, int at) {                             // the i-th load of stage s, into slot `at`
    unsigned char* slot = wl_lds + at * kSlot;
    const bf16* src = i < LW ? wbase[i < LW ? i : 0] + (size_t)s * 1024 : xbase[i < LW ? 0 : i - LW] + (size_t)s * 64;
    unsigned char* dst = i < LW ? slot + min(wave + 4 * i, NB * 2 - 1) * 1024 : slot + NB * 2048 + min(wave + 4 * (i - LW), XT * 2 - 1) * 1024;
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src, (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
  };

  const int wm = wave / WN, wn = wave % WN, r = lane & 15, g = lane >> 4;
  const unsigned char* my_w = wl_lds + wn * NW * 2048 + lane * 16;
  const unsigned char* my_x = wl_lds + NB * 2048 + wm * MW * 2048 + r * 128;
  const int piece[2] = {(g ^ (r & 7)) * 16, ((4 + g) ^ (r & 7)) * 16};
  bf16x8 wf[2][NW], xf[2][MW];
  auto take = [&](int i, int slot, int st, bf16x8* w, bf16x8* x) {     // the i-th operand of a step
    if (i < NW) w[i < NW ? i : 0] = *reinterpret_cast<const bf16x8*>(my_w + slot * kSlot + (i * 2 + st) * 1024);
    else x[i < NW ? 0 : i - NW] = *reinterpret_cast<const bf16x8*>(my_x + slot * kSlot + (i - NW) * 2048 + piece[st]);
  };
  floatx4 acc[MW][NW];
#pragma unroll
  for (int t = 0; t < MW; ++t)
#pragma unroll
    for (int u = 0; u < NW; ++u) acc[t][u] = floatx4{0.f, 0.f, 0.f, 0.f};
  // The compiler does not know the instruction in `multiply` and sets no waits around it.  A wait of our own is between the sums' other accesses
  // and the products only if it owns their registers: their zeros come before this, what is done with the results behind it.
  auto hold_sums = [&] {
#pragma unroll
    for (int t = 0; t < MW; ++t)
#pragma unroll
      for (int u = 0; u < NW; ++u) asm volatile("" : "+a"(acc[t][u]));
  };
  auto multiply = [&](int i, const bf16x8* w, const bf16x8* x) {       // the i-th share of a step's products
#pragma unroll
    for (int q = 0; q < MW * NW; ++q) {
      if (q * Q / (MW * NW) != i) continue;
      floatx4& a = acc[q / NW][q % NW];
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(a) : "v"(w[q % NW]), "v"(x[q / NW]));
    }
  };

#pragma unroll
  for (int s = 0; s < R; ++s)
#pragma unroll
    for (int i = 0; i < L; ++i) issue(i, min(s, n - 1), s);
  wait_loads_but<(R - 1) * L>();
  asm volatile("s_barrier" ::: "memory");
#pragma unroll
  for (int i = 0; i < F; ++i) take(i, 0, 0, wf[0], xf[0]);
  hold_sums();
  asm volatile("s_nop 15");                       // (the sums' zeros are written before an instruction that the compiler does not know reads them)
  int slot = 0;
#pragma unroll 1
  for (int s = 0; s < n; ++s) {
#pragma unroll
    for (int i = 0; i < Q; ++i) {
#pragma unroll
      for (int j = 2 * i; j < 2 * i + 2; ++j)
        if (j < F) take(j, slot, 1, wf[1], xf[1]);
      multiply(i, wf[0], xf[0]);
      __builtin_amdgcn_sched_barrier(0);
    }
    wait_loads_but<(R - 2) * L>();                                     // stage s + 1 has landed,
    __builtin_amdgcn_s_waitcnt(0xC07F);                                // and this wavefront has read the last of stage s (lgkmcnt(0))
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    const int next = slot + 1 == R ? 0 : slot + 1, ahead = min(s + R, n - 1);   // (past the last stage: that one again, into a slot nobody reads)
#pragma unroll
    for (int i = 0; i < Q; ++i) {
#pragma unroll
      for (int j = 2 * i; j < 2 * i + 2; ++j)
        if (j < F) take(j, next, 0, wf[0], xf[0]);
      if (i < L) issue(i, ahead, slot);
      multiply(i, wf[1], xf[1]);
      __builtin_amdgcn_sched_barrier(0);
    }
    slot = next;
  }
  wait_loads_but<0>();
  asm volatile("s_nop 15\n s_nop 15");            // (the last products are in their registers)
  hold_sums();

  finish<EPI, MW, NW>(p, acc, row0 + wm * MW * 16, nb * NB + wn * NW, lane);
}

// 16 bytes a lane from a buffer straight into LDS: a lane's own offset and one that all lanes share.
__device__ __forceinline__ void load_to_lds(__amdgpu_buffer_rsrc_t from, int lane_at, int at, unsigned char* to) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(from, (__attribute__((address_space(3))) void*)to, 16, lane_at, at, 0, 0);
}

// The same for tiles of up to 320 x 256 and 256 x 352 outputs.  Where the kernel above stopped there (256 x 192, 2048 rows of 11264 x 2048, cycles a stage of
// 64 columns): 1,536 of products, 1,955 in all.  Two stages of 57 KB were all that LDS holds, so every stage's loads were waited for before the next
// ones were asked for (1,790 cycles for them alone); one wavefront a SIMD issues nothing else while it issues a load (15 cycles each), and
// a vector instruction in eight cycles at best, so that the activation behind took 23,000 of 135,000 cycles.  Here
//   * eight wavefronts, two a SIMD, as WM x 8 / WM over the tile, each with MW tiles of 16 rows x NW blocks of 16 weight rows: the activation takes
//     half as long, and one issues while the other multiplies;
//   * weights come step by step (32 columns) through a ring of RW places of their own, rows in stages of 64 columns (whole lines) through RX: a step's
//     weights are asked for RW - 1 steps ahead, rows 2 RX - 2 or one less, and the loads of a step follow each other without a gap;
//   * operands of weights are read two groups of products ahead into four places in turn, operands of rows are held twice;
//   * loads go through buffers whose moving part is scalar: one register a lane for all weights and one for each load of rows.
// What bounds it now is power: 256 x 352 takes 1,590 cycles a step (1,408 of products) at 1.85 to 2.0 GHz, and the form of it with four wavefronts and 13 % more
// cycles ran as long at 9 % more clock.  2048 rows of 11264 x 2048, with SiLU: 72 us (1.31 PFLOP/s; 97.7 in two rounds of 256 x 192 above, 94 in the
// library with the activation behind); 777 rows 36 (40.6, 45), 1024 rows 41 (46.5, 56); 2048 / 8192 rows of 16384 x 2048 106 / 423 (library 122 / 483).  Plain: 2048 rows of 8512 x 2048 in 256 x 288 60 (library 79), 1178 of 32000 x 2048
// with float results in 256 x 320 146 (168).
template <int EPI, int WM, int MW, int NW, int RW, int RX>
__global__ __launch_bounds__(512, 2) void big_linear_kernel(WideParams p) {
  constexpr int WN = 8 / WM, NB = WN * NW, XT = WM * MW;
  constexpr int kW = NB * 1024, kX = XT * 2048;                        // bytes of a step's weights, of a stage's rows
  constexpr int LW = (NB + 3) / 4, LX = (XT * 2 + 3) / 4;              // loads of a step's weights, of a stage's rows, that a wavefront which makes them has
  extern __shared__ __attribute__((aligned(16))) unsigned char wl_lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = blockIdx.x / (8 * p.m_blocks), in_group = blockIdx.x - group * 8 * p.m_blocks, across = min(8, p.n_blocks - group * 8);
  const int nb = group * 8 + in_group % across, row0 = in_group / across * (XT * 16);
  const int n = p.ksteps;                                              // (even)

  const unsigned wbytes = (unsigned)min(NB, p.weight_blocks - nb * NB) * (unsigned)n * 1024u;
  const __amdgpu_buffer_rsrc_t wsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(p.wt + (size_t)nb * NB * p.ksteps * 512), 0, (int)wbytes, 0x00027000);
  const unsigned xbytes = ((unsigned)(min(XT * 16, p.M - row0) - 1) * (unsigned)p.ldx + (unsigned)n * 32u) * 2u;
  const __amdgpu_buffer_rsrc_t xsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(p.x + (size_t)row0 * p.ldx), 0, (int)xbytes, 0x00027000);
  const int xr = lane >> 3, xg = (lane & 7) ^ xr;                      // a load: 8 rows x 128 bytes, the row's pieces in XOR-ed order
  const int wlane = lane * 16;
  int xlane[LX];
#pragma unroll
  for (int i = 0; i < LX; ++i) xlane[i] = (min(min((wave & 3) + 4 * i, XT * 2 - 1) * 8 + xr, p.M - 1 - row0) * p.ldx + xg * 8) * 2;   // rows past the end repeat the last one
  const int wblock = p.ksteps * 1024, wlast = p.weight_blocks - 1 - nb * NB;    // bytes of a block of weight rows, the last one that there is
  auto issue_w = [&](int i, int t, int at) {                           // the i-th load of step t's weights, into place `at` (a share that is one short repeats its last one)
    const int bb = min((wave & 3) + 4 * i, NB - 1);
    load_to_lds(wsrc, wlane, min(bb, wlast) * wblock + t * 1024, wl_lds + at * kW + bb * 1024);
  };
  auto issue_x = [&](int i, int s, int at) {
    const int bb = min((wave & 3) + 4 * i, XT * 2 - 1);
    load_to_lds(xsrc, xlane[i], s * 128, wl_lds + RW * kW + at * kX + bb * 1024);
  };

  const int wm = wave / WN, wn = wave % WN, r = lane & 15, g = lane >> 4;
  const unsigned char* my_w = wl_lds + wn * NW * 1024 + lane * 16;
  const unsigned char* my_x = wl_lds + RW * kW + wm * MW * 2048 + r * 128;
  const int piece[2] = {(g ^ (r & 7)) * 16, ((4 + g) ^ (r & 7)) * 16};
  bf16x8 wf[4], xf[2][MW];
  // The place of operand u of an even or odd step: any three in a row, and the last two and first two of a step, lie apart.
  static_assert(NW >= 2 && NW != 5, "four places");
  auto place = [](int u, int st) { return NW == 2 ? st * 2 + u : NW % 3 == 0 ? u % 3 : NW % 3 == 1 ? (u < 4 ? u : (u - 4) % 3) : u < 8 ? u % 4 : (u - 8) % 3; };
  constexpr int kHeld = 32;                                            // blocks of sums in accumulation registers, which are half of all
  floatx4 acc[MW][NW];
#pragma unroll
  for (int t = 0; t < MW; ++t)
#pragma unroll
    for (int u = 0; u < NW; ++u) acc[t][u] = floatx4{0.f, 0.f, 0.f, 0.f};
  auto hold_sums = [&] {                                               // (as above)
#pragma unroll
    for (int u = 0; u < NW; ++u)
#pragma unroll
      for (int t = 0; t < MW; ++t) {
        if (u * MW + t < kHeld) asm volatile("" : "+a"(acc[t][u]));
        else asm volatile("" : "+v"(acc[t][u]));
      }
  };
  auto multiply = [&](int u, int i, int st) {
    if (u * MW + i < kHeld) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][u]) : "v"(wf[place(u, st)]), "v"(xf[st][i]));
    else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc[i][u]) : "v"(wf[place(u, st)]), "v"(xf[st][i]));
  };
  // Wavefronts 0 to 3 ask for rows, 4 to 7 for weights: a wavefront's loads return in the order in which they were asked for, and rows, which come from the
  // L2, would wait behind weights that come from memory for steps much further on.  Period t lies between the barriers of steps t and t + 1 and
  // asks for the weights of step t + RW and, if t is odd, for the rows of stage (t - 1) / 2 + RX (with three places and more: for half of them, and period t + 1
  // for the others), dealt out over the NW groups of products that it has.
  // Step t's barrier, behind the third group from its end: everybody has read step t's operands; step t + 1's weights and rows have landed.
  constexpr bool kSpread = RX > 2;
  constexpr int kWeightsBehind = (RW - 2) * LW, kRowsBehind = (RX - 2) * LX;     // loads that may be under way then
  static_assert(RW >= 3 && RX >= 2 && kWeightsBehind + LW < 64 && kRowsBehind + LX < 64, "vmcnt has six bits");
  auto steps = [&](auto weights) __attribute__((always_inline)) {
    constexpr bool W = decltype(weights)::value;
    auto issue_period = [&](bool odd, int q, int ws, int wat, int xs, int xat) __attribute__((always_inline)) {
      if (!W && !odd && !kSpread) return;
#pragma unroll
      for (int j = 0; j < (W ? LW : LX); ++j) {
        if (W ? j * NW / LW != q : kSpread ? j * 2 * NW / LX != (odd ? q : q + NW) : j * NW / LX != q) continue;
        if (W) issue_w(j < LW ? j : 0, ws, wat);
        else issue_x(j < LX ? j : 0, xs, xat);
      }
    };
    auto barrier = [&](int st) __attribute__((always_inline)) {
      if (W) wait_loads_but<kWeightsBehind>();
      else if (st) wait_loads_but<kRowsBehind>();
      __builtin_amdgcn_s_waitcnt(0xC07F);                              // (lgkmcnt(0): this wavefront has read the last of step t's operands)
      asm volatile("s_barrier" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
    };
    if (W) {
#pragma unroll
      for (int t = 0; t < RW - 1; ++t)
#pragma unroll
        for (int i = 0; i < LW; ++i) issue_w(i, min(t, n - 1), t);
    } else {
#pragma unroll
      for (int s = 0; s < RX - 1; ++s)
#pragma unroll
        for (int i = 0; i < LX; ++i) issue_x(i, min(s, n / 2 - 1), s);
    }
    hold_sums();                                                       // (their zeros are written while the loads travel)
    __builtin_amdgcn_sched_barrier(0);
    wait_loads_but<W ? kWeightsBehind : kRowsBehind>();
    asm volatile("s_barrier" ::: "memory");
#pragma unroll
    for (int t = 0; t < MW; ++t) xf[0][t] = *reinterpret_cast<const bf16x8*>(my_x + t * 2048 + piece[0]);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      wf[place(u, 0)] = *reinterpret_cast<const bf16x8*>(my_w + u * 1024);
      issue_period(true, u, min(RW - 1, n - 1), RW - 1, min(RX - 1, n / 2 - 1), RX - 1);
    }
    asm volatile("s_nop 15");                     // (the sums' zeros are written before an instruction that the compiler does not know reads them)
    int wat = 0, xat = 0, wbefore = RW - 1, xbefore = RX - 1;          // places of step t, of its stage, of those before
#pragma unroll 1
    for (int t = 0; t < n; t += 2) {
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const int wnext = wat + 1 == RW ? 0 : wat + 1, xnext = xat + 1 == RX ? 0 : xat + 1;
        const unsigned char *w0 = my_w + wat * kW, *w1 = my_w + wnext * kW, *x1 = my_x + (st ? xnext : xat) * kX + piece[st ^ 1];
        if (NW == 2) barrier(st);
#pragma unroll
        for (int u = 0; u < NW; ++u) {
          if (u < NW - 2) {
            wf[place(u + 2, st)] = *reinterpret_cast<const bf16x8*>(w0 + (u + 2) * 1024);
            issue_period(st == 0, u + 2, min(t + st - 1 + RW, n - 1), wbefore, min((t >> 1) - 1 + RX, n / 2 - 1), xbefore);
          } else {
            wf[place(u + 2 - NW, st ^ 1)] = *reinterpret_cast<const bf16x8*>(w1 + (u + 2 - NW) * 1024);
#pragma unroll
            for (int i = 0; i < MW; ++i)
              if (i * 2 / MW == u + 2 - NW) xf[st ^ 1][i] = *reinterpret_cast<const bf16x8*>(x1 + i * 2048);
            // (past the end: the last ones again, into places that nobody reads)
            issue_period(st == 1, u + 2 - NW, min(t + st + RW, n - 1), wat, min((t >> 1) + st - 1 + RX, n / 2 - 1), st ? xat : xbefore);
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < MW; ++i) multiply(u, i, st);
          __builtin_amdgcn_sched_barrier(0);
          if (u == NW - 3) barrier(st);
        }
        wbefore = wat;
        wat = wnext;
        if (st) xbefore = xat, xat = xnext;
      }
    }
  };
  if (wave >= 4) steps(std::true_type{});
  else steps(std::false_type{});
  wait_loads_but<0>();
  asm volatile("s_nop 15\n s_nop 15");            // (the last products are in their registers)
  hold_sums();
  if constexpr (EPI != WL_GATED) {
    finish<EPI, MW, NW>(p, acc, row0 + wm * MW * 16, nb * NB + wn * NW, lane);
    return;
  }
  // Gated results go through LDS, a wavefront's 16 rows at a time, so that a store writes 16 bytes a lane along the rows.
  constexpr int kRowBytes = NW * 16 + 16, kMine = 16 * kRowBytes, kHalf = (NW + 1) / 2, kSlow = 2 * kHalf * 64 * 8;      // (rows 16 bytes apart modulo the banks)
  static_assert(8 * (kMine + kSlow) <= RW * kW + RX * kX, "the rings hold the results");
  asm volatile("s_barrier" ::: "memory");         // (everybody's operands are read and loads have landed)
  unsigned char* mine = wl_lds + wave * kMine;
  unsigned char* at = mine + r * kRowBytes + ((g & 1) * 4 + (g >> 1) * 2) * 2;
  f32x2* slow = reinterpret_cast<f32x2*>(wl_lds + 8 * kMine + wave * kSlow) + lane;
  const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(p.out, 0, (int)((unsigned)p.M * (unsigned)p.ldo * 2u), 0x00027000);
  const int c0 = (nb * NB + wn * NW) * 8, m0 = row0 + wm * MW * 16;
  auto activate = [&](const floatx4* sums, unsigned char* to, auto count) {      // one row tile's `count` blocks
    constexpr int C = decltype(count)::value;
    float z[2 * C], y[2 * C], quick[2 * C];
#pragma unroll
    for (int u = 0; u < C; ++u) swap_halves(sums[u], z + 2 * u, y + 2 * u);
    if (!quick_gate(z, quick, p.activation)) {                         // one by one, through LDS: a loop that is not unrolled into as many of them
#pragma unroll
      for (int i = 0; i < 2 * C; ++i) slow[i * 64] = f32x2{z[i], quick[i]};
#pragma unroll 1
      for (int i = 0; i < 2 * C; ++i) {
        const float v = slow[i * 64][0];
        if (!(fabsf(v) < quick_limit(p.activation))) slow[i * 64][1] = gate_activation(v, p.activation);
      }
#pragma unroll
      for (int i = 0; i < 2 * C; ++i) quick[i] = slow[i * 64][1];
    }
#pragma unroll
    for (int i = 0; i < 2 * C; ++i) z[i] = quick[i] * y[i];
#pragma unroll
    for (int u = 0; u < C; ++u) *reinterpret_cast<unsigned*>(to + u * 16) = two_bf16(z[2 * u], z[2 * u + 1]);
  };
#pragma unroll
  for (int t = 0; t < MW; ++t) {
    activate(acc[t], at, std::integral_constant<int, kHalf>{});
    activate(acc[t] + kHalf, at + kHalf * 16, std::integral_constant<int, NW - kHalf>{});
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int i = 0; i < (16 * NW + 63) / 64; ++i) {
      const int c = i * 64 + lane, row = c / NW, piece = c - row * NW, left = p.N - (c0 + piece * 8), m = m0 + t * 16 + row;
      const bool is = row < 16 && m < p.M;
      const u32x4 v = *reinterpret_cast<const u32x4*>(mine + min(row, 15) * kRowBytes + piece * 16);
      const int to = (m * p.ldo + c0 + piece * 8) * 2;
      __builtin_amdgcn_raw_buffer_store_b128(v, out, is && left >= 8 ? to : -1, 0, 0);
      if (p.N & 7) __builtin_amdgcn_raw_buffer_store_b64(u32x2{v[0], v[1]}, out, is && left == 4 ? to : -1, 0, 0);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
}

template <int EPI, int WM, int MW, int NW, int R>
static int launch_wide(WideParams p, int weight_rows, hipStream_t stream) {
  constexpr int kRows = 16 * WM * MW, kWeights = 64 / WM * NW;
  constexpr size_t lds = (size_t)R * (WM * MW + 4 / WM * NW) * 2048;
  static_assert(lds <= 160 * 1024, "LDS of one compute unit");
  auto kernel = wide_linear_kernel<EPI, WM, MW, NW, R>;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return (int)e;
  p.n_blocks = (weight_rows + kWeights - 1) / kWeights;
  p.m_blocks = (p.M + kRows - 1) / kRows;
  if ((long)p.n_blocks * p.m_blocks > 0x7fffffffL / 256) return -2;
  hipLaunchKernelGGL(kernel, dim3(p.n_blocks * p.m_blocks), dim3(256), lds, stream, p);
  return (int)hipGetLastError();
}

template <int EPI, int WM, int MW, int NW, int RW, int RX>
static int launch_big(WideParams p, int weight_rows, hipStream_t stream) {
  constexpr int kRows = 16 * WM * MW, kWeights = 128 / WM * NW;
  constexpr size_t lds = (size_t)RW * (8 / WM * NW) * 1024 + (size_t)RX * (WM * MW) * 2048;
  static_assert(lds <= 160 * 1024, "LDS of one compute unit");
  if (p.ldx >= 1 << 21 || p.ksteps >= 1 << 16) return -2;        // (a tile's 320 rows and 352 weight rows by 32-bit offsets)
  auto kernel = big_linear_kernel<EPI, WM, MW, NW, RW, RX>;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return (int)e;
  p.n_blocks = (weight_rows + kWeights - 1) / kWeights;
  p.m_blocks = (p.M + kRows - 1) / kRows;
  if ((long)p.n_blocks * p.m_blocks > 0x7fffffffL / 512) return -2;
  hipLaunchKernelGGL(kernel, dim3(p.n_blocks * p.m_blocks), dim3(512), lds, stream, p);
  return (int)hipGetLastError();
}

template <int EPI>
static int launch_tile(const WideParams& p, int weight_rows, int rows, int weights, hipStream_t stream) {
  switch (rows * 1000 + weights) {
    case 64064: return launch_wide<EPI, 2, 2, 2, 4>(p, weight_rows, stream);
    case 64128: return launch_wide<EPI, 2, 2, 4, 4>(p, weight_rows, stream);
    case 96096: return launch_wide<EPI, 2, 3, 3, 4>(p, weight_rows, stream);
    case 80128: return launch_wide<EPI, 1, 5, 2, 4>(p, weight_rows, stream);
    case 96128: return launch_wide<EPI, 2, 3, 4, 4>(p, weight_rows, stream);
    case 128128: return launch_wide<EPI, 2, 4, 4, 4>(p, weight_rows, stream);
    case 128160: return launch_wide<EPI, 2, 4, 5, 4>(p, weight_rows, stream);
  }
  if constexpr (EPI != WL_ROPE_KV) {                                   // (in one round where tiles of 256 x 256 need two: ops.wide_plain_plan)
    switch (rows * 1000 + weights) {
      case 256288: return launch_big<EPI, 4, 4, 9, 4, 2>(p, weight_rows, stream);
      case 256320: return launch_big<EPI, 4, 4, 10, 4, 2>(p, weight_rows, stream);
      case 256352: return launch_big<EPI, 4, 4, 11, 4, 2>(p, weight_rows, stream);
      case 320256: return launch_big<EPI, 4, 5, 8, 4, 2>(p, weight_rows, stream);
    }
  }
  if constexpr (EPI == WL_GATED) {
    switch (rows * 1000 + weights) {
      case 160256: return launch_big<EPI, 2, 5, 4, 5, 3>(p, weight_rows, stream);
      case 192128: return launch_big<EPI, 4, 3, 4, 10, 3>(p, weight_rows, stream);
      case 192192: return launch_big<EPI, 4, 3, 6, 5, 3>(p, weight_rows, stream);
      case 192256: return launch_big<EPI, 4, 3, 8, 4, 3>(p, weight_rows, stream);
      case 224192: return launch_big<EPI, 2, 7, 3, 4, 3>(p, weight_rows, stream);
      case 224256: return launch_big<EPI, 2, 7, 4, 4, 3>(p, weight_rows, stream);
      case 256128: return launch_big<EPI, 4, 4, 4, 6, 3>(p, weight_rows, stream);
      case 256192: return launch_big<EPI, 4, 4, 6, 4, 3>(p, weight_rows, stream);
      case 256224: return launch_big<EPI, 4, 4, 7, 5, 2>(p, weight_rows, stream);
      case 256256: return launch_big<EPI, 4, 4, 8, 4, 2>(p, weight_rows, stream);
      case 288128: return launch_big<EPI, 2, 9, 2, 6, 3>(p, weight_rows, stream);
      case 320128: return launch_big<EPI, 4, 5, 4, 4, 3>(p, weight_rows, stream);
    }
  }
  return -3;
}

// `rows`, `weights`: the tile, one of the forms above.  `weight_blocks`: blocks of 16 rows that the tiled matrix holds.  K a multiple of 64.
PLLM_API int pllm_wide_linear(int epi, const void* x, int ldx, const void* wt, void* out, int ldo, int M, int N, int K, int weight_blocks, int rows, int weights,
                              const int* positions, const float* cos_t, const float* sin_t, const int* slots, void* k_pages, void* v_pages, int num_heads,
                              int num_kv_heads, int head_dim, int block_size, int activation, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || K % 64 || N % 4 || (ldo & 3) || (reinterpret_cast<uintptr_t>(out) & 15) || (unsigned long)M * ldo >= (1ul << 29) || (ldx & 7) || (reinterpret_cast<uintptr_t>(x) & 15) || weight_blocks <= 0 || activation < 0) return -2;
  const int weight_rows = epi == WL_GATED ? 2 * ((N + 7) / 8 * 8) : N;
  if ((long)weight_blocks * 16 < weight_rows) return -2;
  const WideParams p{(const bf16*)x, (const bf16*)wt, out, ldx, ldo, M, N, K / 32, weight_blocks, 0, 0, activation, num_heads, num_kv_heads, head_dim, block_size,
                     positions, slots, cos_t, sin_t, (bf16*)k_pages, (bf16*)v_pages};
  switch (epi) {
    case WL_BF16: return launch_tile<WL_BF16>(p, weight_rows, rows, weights, stream);
    case WL_F32: return launch_tile<WL_F32>(p, weight_rows, rows, weights, stream);
    case WL_GATED: return activation < PLLM_ACT_COUNT ? launch_tile<WL_GATED>(p, weight_rows, rows, weights, stream) : -2;
    case WL_ROPE_KV:
      if (head_dim <= 0 || (head_dim % 16) || !slots || !k_pages || !v_pages || !positions || N != (num_heads + 2 * num_kv_heads) * head_dim || block_size <= 0 || (ldo & 3)) return -2;
      return launch_tile<WL_ROPE_KV>(p, weight_rows, rows, weights, stream);
  }
  return -3;
}
