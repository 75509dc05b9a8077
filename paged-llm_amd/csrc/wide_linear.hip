// Products of prompt steps: y = x W^T for bfloat16 rows and a tiled weight matrix (ops.tile_weight), in tiles of 64 x 64 to 256 x 192
// outputs, one workgroup of four wavefronts a tile, with bfloat16 or float results, act(gate) * up, or the rotation of q and k
// with the write of k and v into their cache pages behind.
//
// What bounds it: the matrix cores at the clock that they hold under such a load (1.3 to 1.4 PFLOP/s over the chip with nothing else in the
// kernel), and for tiles of 128 x 128 and less a compute unit's way to the L2 (26 to 45 bytes a clock).  So every other
// instruction has to hide behind the products, and one wavefront per SIMD with up to 512 registers does that:
//   * Stages of 64 columns lie in LDS, R of them, filled by global_load_lds (16 bytes a lane, no registers in between): weights in whole
//     kilobytes in operand order, rows in pieces of 128 bytes in an order that spreads the banks.
//   * A stage's columns are two steps of 32.  While the products of one step run, the operands of the next come from LDS; in the middle of
//     a stage, behind the only barrier, its slot is free and the loads of the stage R ahead are issued.
//   * Loads, LDS reads and products are dealt out evenly in the source and kept there: the loads of a stage in front of its
//     products hold up the wavefront until the memory pipe has taken them all (256 x 192 at 2048 x 11264 x 2048: 119 us, dealt out 95).
//   * The sums are held in the accumulation registers by the instruction's own operand constraint: left to itself the compiler moves
//     them to and fro (96 to 248 moves a stage).
// Measured (us, weights from memory; in brackets the library's product, with the kernel behind it where there is one): 896 rows x 2048 x 2048 14.0 (16.4),
// 512 x 1024 x 1024 5.7 (8.4), 2048 x 2048 x 4096 39.5 (40.4), gated 512 rows of 5632 x 1024 13.4 (20.6), 320 / 777 / 1024 rows of 11264 x 2048 25.4 /
// 40.6 / 46.5 (33.0 / 45.4 / 58.6).
// Which tile a product takes, and whether it comes here, is the host's choice (ops.wide_linear_plan, ops.wide_rotary_plan).
// An output is one chain in ascending k whatever its tile.
// moe_wide.hip has the same stages, waits and held sums for the experts' products: what is mended in one belongs in the other.
#include "common.h"

using namespace pllm;

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float floatx4;
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

// exp(x) for |x| < 87 from the instruction for 2^x: x / ln 2 as a rounded product and what the rounding left, the whole part n put into the
// exponent.
__device__ __forceinline__ float exp_near(float x) {
#pragma clang fp contract(off)
  const float t = x * 1.44269504f, n = __builtin_rintf(t), left = fmaf(x, 1.9259629911e-8f, fmaf(x, 1.44269504f, -t));
  return __builtin_ldexpf(__builtin_amdgcn_exp2f((t - n) + left), (int)n);
}

// act(z) times y in place of z, for the results of a lane that lie in one row.  SiLU from the quotient's first value corrected once, which leaves the
// error that expf and a division have (relative to 64 bits, over z from -87 to 87: RMS 3.6e-8, at most 1.8e-7) at half of their
// instructions, without a branch inside (there is one wavefront per SIMD: what one result waits for, the others fill).
template <int COUNT>
__device__ __forceinline__ void gate(float (&z)[COUNT], const float (&y)[COUNT], int act) {
  if (act != PLLM_ACT_SILU) {
#pragma unroll
    for (int i = 0; i < COUNT; ++i) z[i] = gate_activation(z[i], act) * y[i];
    return;
  }
  float fast[COUNT];
  bool near = true;
#pragma unroll
  for (int i = 0; i < COUNT; ++i) {
    const float d = 1.f + exp_near(-z[i]), r = __builtin_amdgcn_rcpf(d), q = z[i] * r;
    fast[i] = fmaf(fmaf(-q, d, z[i]), r, q);
    near = near && fabsf(z[i]) < 87.f;                                 // (infinities, NaN and 1 / (1 + exp(-z)) below the normal numbers are not)
  }
  if (!__all(near)) {
#pragma unroll
    for (int i = 0; i < COUNT; ++i)
      if (!(fabsf(z[i]) < 87.f)) fast[i] = gate_activation(z[i], PLLM_ACT_SILU);
  }
#pragma unroll
  for (int i = 0; i < COUNT; ++i) z[i] = fast[i] * y[i];
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

  // A lane's four sums are four weight rows (4 g .. 4 g + 3 of the block) of input row r of the tile.  Stores go through a buffer that drops what
  // lies past its end, so that no store has a branch of its own (with branches the end of 128 x 128 took 3 us longer).
  const int row_bytes = p.ldo * (EPI == WL_F32 ? 4 : 2);
  const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(p.out, 0, (int)((unsigned)p.M * (unsigned)row_bytes), 0x00027000);
  // Products that take two weight rows: rows 8-15 of a block (the lanes 32 further on) are the partners of rows 0-7.  The halves change places so
  // that lanes 0-31 have rows 4 g, 4 g + 1 and lanes 32-63 rows 4 g + 2, 4 g + 3, with their partners.
  const int pair_row = (g & 1) * 4 + (g >> 1) * 2;
  auto halves = [&](const floatx4& a, float* one, float* other) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(a[i]), __float_as_uint(a[i + 2]), false, false);
      one[i] = __uint_as_float(x[0]);
      other[i] = __uint_as_float(x[1]);
    }
  };
  auto two = [](float x, float y) {
    struct { bf16 v[2]; } o{{__float2bfloat16(x), __float2bfloat16(y)}};
    return __builtin_bit_cast(unsigned, o);
  };
#pragma unroll
  for (int t = 0; t < MW; ++t) {
    const int m = row0 + (wm * MW + t) * 16 + r;
    const int at_row = m * row_bytes;
    int pos = 0, slot_kv = -1;
    if (EPI == WL_ROPE_KV && m < p.M) {
      pos = p.positions[m];
      slot_kv = p.slots[m];
    }
    if constexpr (EPI == WL_GATED) {
      float z[2 * NW], y[2 * NW];
#pragma unroll
      for (int u = 0; u < NW; ++u) halves(acc[t][u], z + 2 * u, y + 2 * u);
      gate(z, y, p.activation);
#pragma unroll
      for (int u = 0; u < NW; ++u) {
        const int c = (nb * NB + wn * NW + u) * 8 + pair_row;
        __builtin_amdgcn_raw_buffer_store_b32(two(z[2 * u], z[2 * u + 1]), out, c < p.N && m < p.M ? at_row + 2 * c : -1, 0, 0);
      }
      continue;
    }
    const int page = EPI == WL_ROPE_KV && slot_kv >= 0 ? slot_kv / p.block_size : 0, off = slot_kv - page * p.block_size;
#pragma unroll
    for (int u = 0; u < NW; ++u) {
      const floatx4 a = acc[t][u];
      const int unit = nb * NB + wn * NW + u;
      if constexpr (EPI == WL_F32) {
        const int c = unit * 16 + g * 4;
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, a), out, c < p.N && m < p.M ? at_row + 4 * c : -1, 0, 0);
      } else if constexpr (EPI == WL_BF16) {
        const int c = unit * 16 + g * 4;
        __builtin_amdgcn_raw_buffer_store_b64(u32x2{two(a[0], a[1]), two(a[2], a[3])}, out, c < p.N && m < p.M ? at_row + 2 * c : -1, 0, 0);
      } else {
        float x[2], y[2];
        halves(a, x, y);
        const int d = p.head_dim, half = d >> 1, per_head = half >> 3, nh = p.num_heads, nkv = p.num_kv_heads;
        const int head = unit / per_head, ri = (unit - head * per_head) * 8 + pair_row;
        if (head >= nh + 2 * nkv) continue;
        if (head < nh + nkv) {
          f32x2 cs{1.f, 1.f}, sn{0.f, 0.f};
          if (p.cos_t) {
            cs = *reinterpret_cast<const f32x2*>(p.cos_t + (size_t)pos * half + ri);
            sn = *reinterpret_cast<const f32x2*>(p.sin_t + (size_t)pos * half + ri);
          }
          float lo[2], hi[2];
#pragma unroll
          for (int i = 0; i < 2; ++i)
            rotate_pair(__bfloat162float(__float2bfloat16(x[i])), __bfloat162float(__float2bfloat16(y[i])), cs[i], sn[i], lo[i], hi[i]);
          if (head < nh) {
            const int at = m < p.M ? at_row + 2 * (head * d + ri) : -1;
            __builtin_amdgcn_raw_buffer_store_b32(two(lo[0], lo[1]), out, at, 0, 0);
            __builtin_amdgcn_raw_buffer_store_b32(two(hi[0], hi[1]), out, m < p.M ? at + 2 * half : -1, 0, 0);
          } else if (slot_kv >= 0) {
            bf16* dst = p.k_pages + (((size_t)page * nkv + (head - nh)) * p.block_size + off) * d + ri;
            *reinterpret_cast<unsigned*>(dst) = two(lo[0], lo[1]);
            *reinterpret_cast<unsigned*>(dst + half) = two(hi[0], hi[1]);
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
  if constexpr (EPI == WL_GATED) {                                     // (plain products of so many outputs stay with the library)
    switch (rows * 1000 + weights) {
      case 192192: return launch_wide<EPI, 2, 6, 6, 3>(p, weight_rows, stream);
      case 160256: return launch_wide<EPI, 2, 5, 8, 3>(p, weight_rows, stream);
      case 224192: return launch_wide<EPI, 2, 7, 6, 2>(p, weight_rows, stream);
      case 256192: return launch_wide<EPI, 2, 8, 6, 2>(p, weight_rows, stream);
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
