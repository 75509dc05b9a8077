// The experts' products of prompt steps (moe.hip: the forms, the sorted pairs and their tiles) in tiles of 64 to 192 rows of one expert x 128 or 256
// weight rows, one workgroup of four wavefronts a tile, where K is a multiple of 64.
//
// The structure is that of wide_linear.hip (what is mended in one belongs in the other), and so are the reasons: one wavefront per SIMD with up to 512 registers, stages of 64 columns in
// LDS filled by global_load_lds, R of them, the operands of a step of 32 columns read while the products of the step before it run, loads, reads
// and products dealt out evenly, the sums held in the accumulation registers.  Rows and weights both come as pieces of 8 rows x 128 bytes
// whose eight 16-byte parts lie XOR-ed by the row.
//
// What bounds it: as there a compute unit's way to the L2 and the matrix cores' clock, and the rows that a tile has for nothing: with 2 of 8 experts
// 1,178 tokens are 295 rows an expert, three tiles of 128 (384 rows) or two of 160.  So the host chooses the tile's rows by the expected
// number of tiles and rounds of workgroups (ops.moe_wide_plan, with what was measured against the staged kernel).  A round of 160 x 256 takes 50 us at K =
// 2,048 and 30 at 1,024 (20 and 13 in the matrix cores), 59 and 38 with GELU behind it.
// The sums run over ascending k in one accumulator per output, in steps of 32: the bits of the staged kernel.
#include "common.h"

using namespace pllm;

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float floatx4;
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

enum { kFormDown = 0, kFormGated = 1, kFormPlain = 2 };

struct MoeWide {
  const bf16 *rows_in, *w;
  void* out;
  const int *tiles, *sorted_pair;
  const float* pair_scale;
  int ld_in, ld_out, max_tiles, n_blocks, top, n_out, K, act;
};

template <int N_>
__device__ __forceinline__ void wait_loads_but() {   // until at most N_ of this wavefront's loads are still under way
  static_assert(N_ >= 0 && N_ < 64, "vmcnt has six bits");
  __builtin_amdgcn_s_waitcnt((N_ & 0xf) | ((N_ >> 4) << 14) | 0x0f70);
}

// Wavefronts WM x 4 / WM, each with MW tiles of 16 rows x NW blocks of 16 weight rows.
template <int FORM, int WM, int MW, int NW, int R>
__global__ __launch_bounds__(256, 1) void moe_wide_kernel(MoeWide p) {
  constexpr bool GATED = FORM == kFormGated, FIRST = FORM != kFormDown;
  constexpr int WN = 4 / WM, NB = WN * NW, XT = WM * MW, kOutputs = GATED ? NB * 8 : NB * 16;
  constexpr int kSlot = (NB + XT) * 2048;                              // bytes of a stage: two steps of every block and tile
  constexpr int LW = (NB * 2 + 3) / 4, LX = (XT * 2 + 3) / 4, L = LW + LX, F = MW + NW;   // a wavefront's loads of a stage, its operands of a step
  constexpr int Q = L > F ? L : F;                                     // shares that a step is dealt out in
  static_assert(!GATED || NW % 2 == 0, "a wavefront has a gate's block and its up block");
  extern __shared__ __attribute__((aligned(16))) unsigned char mw_lds[];
  const int group = blockIdx.x / (8 * p.max_tiles), in_group = blockIdx.x - group * 8 * p.max_tiles, across = min(8, p.n_blocks - group * 8);
  const int tile = in_group / across, n0 = (group * 8 + in_group - tile * across) * kOutputs;
  const int expert = __builtin_amdgcn_readfirstlane(p.tiles[3 * tile]), row0 = __builtin_amdgcn_readfirstlane(p.tiles[3 * tile + 1]);
  const int nrows = __builtin_amdgcn_readfirstlane(p.tiles[3 * tile + 2]);
  if (nrows <= 0) return;                                              // the whole workgroup: no barrier is left behind
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = p.K >> 6;                                              // stages

  const bf16 *wbase[LW], *xbase[LX];                                   // (a share that is one load short repeats its last one)
  const int xr = lane >> 3, xg = ((lane & 7) ^ xr) * 8;                // a load: 8 rows x 128 bytes, the row's pieces in XOR-ed order
  const bf16* we = p.w + (size_t)expert * (GATED ? 2 : 1) * p.n_out * p.K;
#pragma unroll
  for (int i = 0; i < LX; ++i) {                                       // (rows past the tile's last repeat it: never stored)
    const int rr = row0 + min(min(wave + 4 * i, XT * 2 - 1) * 8 + xr, nrows - 1);
    xbase[i] = p.rows_in + (size_t)(FIRST ? p.sorted_pair[rr] / p.top : rr) * p.ld_in + xg;
  }
#pragma unroll
  for (int i = 0; i < LW; ++i) {                                       // (outputs past the last repeat it: never stored)
    const int bb = min(wave + 4 * i, NB * 2 - 1), u = bb >> 1, in_block = (bb & 1) * 8 + xr;
    const int row = GATED ? min(n0 + (u >> 1) * 16 + in_block, p.n_out - 1) + (u & 1) * p.n_out : min(n0 + u * 16 + in_block, p.n_out - 1);
    wbase[i] = we + (size_t)row * p.K + xg;
  }
  auto issue = [&](int i, int s, int at) {                             // the i-th load of stage s, into slot `at`
    unsigned char* slot = mw_lds + at * kSlot;
    const bf16* src = (i < LW ? wbase[i < LW ? i : 0] : xbase[i < LW ? 0 : i - LW]) + (size_t)s * 64;
    unsigned char* dst = i < LW ? slot + min(wave + 4 * i, NB * 2 - 1) * 1024 : slot + NB * 2048 + min(wave + 4 * (i - LW), XT * 2 - 1) * 1024;
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src, (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
  };

  const int wm = wave / WN, wn = wave % WN, r = lane & 15, g = lane >> 4;
  const unsigned char* my_w = mw_lds + wn * NW * 2048 + r * 128;
  const unsigned char* my_x = mw_lds + NB * 2048 + wm * MW * 2048 + r * 128;
  const int piece[2] = {(g ^ (r & 7)) * 16, ((4 + g) ^ (r & 7)) * 16};
  bf16x8 wf[2][NW], xf[2][MW];
  auto take = [&](int i, int slot, int st, bf16x8* w, bf16x8* x) {     // the i-th operand of a step
    if (i < NW) w[i < NW ? i : 0] = *reinterpret_cast<const bf16x8*>(my_w + slot * kSlot + i * 2048 + piece[st]);
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

  // A lane's four sums are four outputs (4 g .. 4 g + 3 of a block) of row r of a tile.  A wavefront turns a tile of 16 rows at a time in its own
  // corner of LDS, so that the activation's code stands there once a tile and not once an output (unrolled over the sums it takes longer to fetch
  // than to run), and rows are stored in whole pieces.  Stores go through a buffer that ends behind the tile's last row.
  constexpr int kStride = NW * 16 + 4, kCols = GATED ? NW * 8 : NW * 16;        // floats of a row there; its outputs
  const int esize = FIRST ? 2 : 4, row_bytes = p.ld_out * esize;
  const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc((char*)p.out + (size_t)row0 * row_bytes, 0, nrows * row_bytes, 0x00027000);
  __syncthreads();                                                     // (everybody has read the last stage)
  float* corner = reinterpret_cast<float*>(mw_lds) + wave * 16 * kStride;
  const int col0 = n0 + wn * kCols;
#pragma unroll
  for (int t = 0; t < MW; ++t) {
    const int m0 = (wm * MW + t) * 16;
    const float scales = (FIRST && p.pair_scale) ? p.pair_scale[p.sorted_pair[row0 + min(m0 + r, nrows - 1)]] : 1.f;    // factors on the pairs' input rows
#pragma unroll
    for (int u = 0; u < NW; ++u) *reinterpret_cast<floatx4*>(corner + r * kStride + u * 16 + 4 * g) = acc[t][u];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");             // (LDS takes a wavefront's accesses in order)
#pragma unroll 1
    for (int i = 4 * lane; i < 16 * kCols; i += 256) {
      const int row = i / kCols, c = i - row * kCols;
      const int at = col0 + c < p.n_out && m0 + row < nrows ? (m0 + row) * row_bytes + (col0 + c) * esize : -1;
      const float* from = corner + row * kStride + (GATED ? (c >> 4) * 32 + (c & 15) : c);
      const floatx4 x = *reinterpret_cast<const floatx4*>(from);
      if constexpr (FIRST) {
        const float ps = __shfl(scales, row);
        struct { bf16 v[4]; } y;
        if constexpr (GATED) {
          const floatx4 up = *reinterpret_cast<const floatx4*>(from + 16);
#pragma unroll
          for (int e = 0; e < 4; ++e) y.v[e] = from_f32<bf16>(gate_activation(x[e] * ps, p.act) * (up[e] * ps));
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) y.v[e] = from_f32<bf16>(row_activation_for_bf16(x[e] * ps, p.act));
        }
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, y), out, at, 0, 0);
      } else {
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, x), out, at, 0, 0);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
}

template <int FORM, int WM, int MW, int NW, int R>
static int launch_moe_wide(MoeWide p, hipStream_t stream) {
  constexpr int kOutputs = 64 / WM * NW / (FORM == kFormGated ? 2 : 1);
  constexpr size_t lds = (size_t)R * (WM * MW + 4 / WM * NW) * 2048;
  static_assert(lds <= 160 * 1024, "LDS of one compute unit");
  auto kernel = moe_wide_kernel<FORM, WM, MW, NW, R>;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return (int)e;
  p.n_blocks = (p.n_out + kOutputs - 1) / kOutputs;
  if ((long)p.n_blocks * p.max_tiles > 0x7fffffffL / 256) return -2;
  hipLaunchKernelGGL(kernel, dim3(p.n_blocks * p.max_tiles), dim3(256), lds, stream, p);
  return (int)hipGetLastError();
}

template <int FORM>
static int launch_form(const MoeWide& p, int rows, int weights, hipStream_t stream) {
  switch (rows * 1000 + weights) {
    case 64128: return launch_moe_wide<FORM, 2, 2, 4, 4>(p, stream);
    case 64256: return launch_moe_wide<FORM, 1, 4, 4, 4>(p, stream);
    case 96128: return launch_moe_wide<FORM, 2, 3, 4, 4>(p, stream);
    case 96256: return launch_moe_wide<FORM, 2, 3, 8, 3>(p, stream);
    case 128128: return launch_moe_wide<FORM, 2, 4, 4, 4>(p, stream);
    case 128256: return launch_moe_wide<FORM, 2, 4, 8, 3>(p, stream);
    case 160128: return launch_moe_wide<FORM, 2, 5, 4, 4>(p, stream);
    case 160256: return launch_moe_wide<FORM, 2, 5, 8, 3>(p, stream);
    case 192128: return launch_moe_wide<FORM, 2, 6, 4, 4>(p, stream);
    case 192256: return launch_moe_wide<FORM, 2, 6, 8, 2>(p, stream);
  }
  return -3;
}

// form, tiles, sorted_pair, top, pair_scale as pllm_moe_expert_gemm takes them (bfloat16); `rows`: the tiles' rows, `weights`: the weight rows of a
// workgroup, one of the forms above.  K a multiple of 64, n_out and ld_out of 4, operands on 16-byte boundaries.
PLLM_API int pllm_moe_expert_wide(int form, const void* rows_in, int ld_in, const void* w, const int* tiles, int max_tiles, int rows, int weights,
                                  const int* sorted_pair, int top, int n_out, int K, void* out, int ld_out, int act, const float* pair_scale,
                                  hipStream_t stream) {
  if (max_tiles <= 0) return 0;
  if (n_out <= 0 || n_out % 4 || ld_out % 4 || K <= 0 || K % 64 || ld_in % 8 || top <= 0 || act < 0 || act >= (form == kFormPlain ? PLLM_ROW_ACT_COUNT : PLLM_ACT_COUNT) || act == PLLM_ROW_ACT_XIELU) return -2;
  if ((reinterpret_cast<uintptr_t>(rows_in) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(out)) & 15 || (long)rows * ld_out >= 1l << 28) return -2;
  const MoeWide p{(const bf16*)rows_in, (const bf16*)w, out, tiles, sorted_pair, pair_scale, ld_in, ld_out, max_tiles, 0, top, n_out, K, act};
  switch (form) {
    case kFormDown: return launch_form<kFormDown>(p, rows, weights, stream);
    case kFormGated: return launch_form<kFormGated>(p, rows, weights, stream);
    case kFormPlain: return launch_form<kFormPlain>(p, rows, weights, stream);
  }
  return -3;
}
