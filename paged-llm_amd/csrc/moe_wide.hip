// The experts' products of prompt steps (moe.hip: the forms, the sorted pairs and their tiles) in tiles of 64 to 192 rows of one expert x 128 or 256
// weight rows, one workgroup of eight wavefronts a tile, where K is a multiple of 64.
//
// The structure is that of wide_linear.hip's kernel with eight wavefronts (what is mended in one belongs in the other), and so are the reasons: two wavefronts
// a SIMD, rows and weights asked for by different ones, operands of weights read two groups of products ahead, the sums held in the accumulation
// registers.  Rows and weights both come as pieces of 8 rows x 128 bytes whose eight 16-byte parts lie XOR-ed by the row, in stages of
// 64 columns, R of them in LDS.
//
// What bounds it: as there a compute unit's way to the L2 and the matrix cores' clock, weights that come from memory beside rows that do not, and the rows
// that a tile has for nothing: with 2 of 8 experts 1,178 tokens are 295 rows an expert, three tiles of 128 (384 rows) or two of 160.  So the host chooses the
// tile's rows by the expected number of tiles and rounds of workgroups (ops.moe_wide_plan, with what was measured against the staged kernel).
// Measured (us, first / down product, weights from memory; in brackets four wavefronts with twice the registers): 2,048 tokens with 2 of 8 plain experts of
// 4,096 at width 2,048 in 160 x 256 94 / 77 (107 / 82), 2 of 8 gated ones of 2,048 86 / 44 (96 / 48), 4 of 16 plain ones of 1,024 at width 1,024 30 / 28 (39 / 30), 1,000
// tokens with 4 of 16 plain ones of 2,048 52 / 51 (60 / 52); 192 x 256, whose two stages are all that LDS holds, 5 % faster and 3 % slower on average.
// The sums run over ascending k in one accumulator per output, in steps of 32: the bits of the staged kernel.
#include "common.h"
#include <type_traits>

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

// Wavefronts WM x 8 / WM, each with MW tiles of 16 rows x NW blocks of 16 weight rows.
template <int FORM, int WM, int MW, int NW, int R>
__global__ __launch_bounds__(512, 2) void moe_wide_kernel(MoeWide p) {
  constexpr bool GATED = FORM == kFormGated, FIRST = FORM != kFormDown;
  constexpr int WN = 8 / WM, NB = WN * NW, XT = WM * MW, kOutputs = GATED ? NB * 8 : NB * 16;
  constexpr int kSlot = (NB + XT) * 2048;                              // bytes of a stage: two steps of every block and tile
  constexpr int LW = (NB * 2 + 3) / 4, LX = (XT * 2 + 3) / 4;          // loads of a stage's weights, of its rows, that a wavefront which makes them has
  static_assert(!GATED || NW % 2 == 0, "a wavefront has a gate's block and its up block");
  extern __shared__ __attribute__((aligned(16))) unsigned char mw_lds[];
  const int group = blockIdx.x / (8 * p.max_tiles), in_group = blockIdx.x - group * 8 * p.max_tiles, across = min(8, p.n_blocks - group * 8);
  const int tile = in_group / across, n0 = (group * 8 + in_group - tile * across) * kOutputs;
  const int expert = __builtin_amdgcn_readfirstlane(p.tiles[3 * tile]), row0 = __builtin_amdgcn_readfirstlane(p.tiles[3 * tile + 1]);
  const int nrows = __builtin_amdgcn_readfirstlane(p.tiles[3 * tile + 2]);
  if (nrows <= 0) return;                                              // the whole workgroup: no barrier is left behind
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = p.K >> 6;                                              // stages
  const int xr = lane >> 3, xg = ((lane & 7) ^ xr) * 8;                // a load: 8 rows x 128 bytes, the row's pieces in XOR-ed order
  const int wm = wave / WN, wn = wave % WN, r = lane & 15, g = lane >> 4;
  const unsigned char* my_w = mw_lds + wn * NW * 2048 + r * 128;
  const unsigned char* my_x = mw_lds + NB * 2048 + wm * MW * 2048 + r * 128;
  const int piece[2] = {(g ^ (r & 7)) * 16, ((4 + g) ^ (r & 7)) * 16};
  bf16x8 wf[4], xf[2][MW];
  // The place of operand u of an even or odd step: any three in a row, and the last two and first two of a step, lie apart.
  static_assert(NW == 2 || NW == 4 || NW == 8, "four places");
  auto place = [](int u, int st) { return NW == 2 ? st * 2 + u : u & 3; };
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
  auto multiply = [&](int u, int i, int st) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][u]) : "v"(wf[place(u, st)]), "v"(xf[st][i]));
  };
  // Wavefronts 0 to 3 ask for rows, 4 to 7 for weights, whose loads take longer and would hold up the rows' behind them.  Stage s's barrier stands in its second
  // step where everybody has read the last of its operands; stage s + 1 has landed then, and the loads of stage s + R are dealt out over the 2 NW groups of
  // products up to the next one (with two slots, where they have to land by then, over the first half of them).
  auto stages = [&](auto weights) __attribute__((always_inline)) {
    constexpr bool W = decltype(weights)::value;
    constexpr int L = W ? LW : LX;
    const bf16* base[L];                                               // (a share that is one load short repeats its last one)
#pragma unroll
    for (int i = 0; i < L; ++i) {
      const int bb = min((wave & 3) + 4 * i, (W ? NB : XT) * 2 - 1);
      if (W) {                                                         // (outputs past the last repeat it: never stored)
        const int u = bb >> 1, in_block = (bb & 1) * 8 + xr;
        const int row = GATED ? min(n0 + (u >> 1) * 16 + in_block, p.n_out - 1) + (u & 1) * p.n_out : min(n0 + u * 16 + in_block, p.n_out - 1);
        base[i] = p.w + ((size_t)expert * (GATED ? 2 : 1) * p.n_out + row) * p.K + xg;
      } else {                                                         // (rows past the tile's last repeat it: never stored)
        const int rr = row0 + min(bb * 8 + xr, nrows - 1);
        base[i] = p.rows_in + (size_t)(FIRST ? p.sorted_pair[rr] / p.top : rr) * p.ld_in + xg;
      }
    }
    auto issue = [&](int i, int s, int at) __attribute__((always_inline)) {      // the i-th load of stage s, into slot `at`
      const int bb = min((wave & 3) + 4 * i, (W ? NB : XT) * 2 - 1);
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(base[i] + (size_t)min(s, n - 1) * 64),
                                       (__attribute__((address_space(3))) void*)(mw_lds + at * kSlot + (W ? 0 : NB * 2048) + bb * 1024), 16, 0, 0);
    };
    constexpr int kBehind = (R - 2) * L, kOver = R == 2 ? NW : 2 * NW;  // loads that may be under way at a barrier; groups that a stage's loads are dealt out over
    auto issue_group = [&](int q, int s, int at) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < L; ++j)
        if (j * kOver / L == q) issue(j, s, at);
    };
    static_assert(R >= 2 && kBehind + L < 64, "vmcnt has six bits");
#pragma unroll
    for (int s = 0; s < R - 1; ++s)
#pragma unroll
      for (int i = 0; i < L; ++i) issue(i, s, s);
    hold_sums();                                                       // (their zeros are written while the loads travel)
    __builtin_amdgcn_sched_barrier(0);
    wait_loads_but<kBehind>();
    asm volatile("s_barrier" ::: "memory");
    constexpr int kAhead = 2;                                          // groups of a period that lie in the stage before
#pragma unroll
    for (int i = 0; i < MW; ++i) xf[0][i] = *reinterpret_cast<const bf16x8*>(my_x + i * 2048 + piece[0]);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      wf[place(u, 0)] = *reinterpret_cast<const bf16x8*>(my_w + u * 2048 + piece[0]);
      issue_group(u, R - 1, R - 1);
    }
    asm volatile("s_nop 15");                     // (the sums' zeros are written before an instruction that the compiler does not know reads them)
    auto barrier = [&]() __attribute__((always_inline)) {
      wait_loads_but<kBehind>();                                       // stage s + 1 has landed,
      __builtin_amdgcn_s_waitcnt(0xC07F);                              // and this wavefront has read the last of stage s (lgkmcnt(0))
      asm volatile("s_barrier" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
    };
    // A period's first two groups are the last two of a stage, behind its barrier; the others are the next stage's.
    int slot = 0, before = R - 1;
#pragma unroll 1
    for (int s = 0; s < n; ++s) {
      const int next = slot + 1 == R ? 0 : slot + 1;
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        if (NW == 2 && st == 1) barrier();
#pragma unroll
        for (int u = 0; u < NW; ++u) {
          if (u < NW - 2) wf[place(u + 2, st)] = *reinterpret_cast<const bf16x8*>(my_w + slot * kSlot + (u + 2) * 2048 + piece[st]);
          else {
            const int from = st ? next : slot;
            wf[place(u + 2 - NW, st ^ 1)] = *reinterpret_cast<const bf16x8*>(my_w + from * kSlot + (u + 2 - NW) * 2048 + piece[st ^ 1]);
#pragma unroll
            for (int i = 0; i < MW; ++i)
              if (i * 2 / MW == u + 2 - NW) xf[st ^ 1][i] = *reinterpret_cast<const bf16x8*>(my_x + from * kSlot + i * 2048 + piece[st ^ 1]);
          }
          // (past the last stage: that one again, into slots that nobody reads)
          if (st == 1 && u >= NW - 2) issue_group(u - (NW - kAhead), s + R, slot);
          else issue_group(st * NW + u + kAhead, s - 1 + R, before);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < MW; ++i) multiply(u, i, st);
          __builtin_amdgcn_sched_barrier(0);
          if (st == 1 && u == NW - 3) barrier();
        }
      }
      before = slot;
      slot = next;
    }
  };
  if (wave >= 4) stages(std::true_type{});
  else stages(std::false_type{});
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
  constexpr int kOutputs = 128 / WM * NW / (FORM == kFormGated ? 2 : 1);
  constexpr size_t lds = (size_t)R * (WM * MW + 8 / WM * NW) * 2048;
  static_assert(lds <= 160 * 1024, "LDS of one compute unit");
  auto kernel = moe_wide_kernel<FORM, WM, MW, NW, R>;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return (int)e;
  p.n_blocks = (p.n_out + kOutputs - 1) / kOutputs;
  if ((long)p.n_blocks * p.max_tiles > 0x7fffffffL / 512) return -2;
  hipLaunchKernelGGL(kernel, dim3(p.n_blocks * p.max_tiles), dim3(512), lds, stream, p);
  return (int)hipGetLastError();
}

template <int FORM>
static int launch_form(const MoeWide& p, int rows, int weights, hipStream_t stream) {
  switch (rows * 1000 + weights) {
    case 64128: return launch_moe_wide<FORM, 2, 2, 2, 4>(p, stream);
    case 64256: return launch_moe_wide<FORM, 2, 2, 4, 4>(p, stream);
    case 96128: return launch_moe_wide<FORM, 2, 3, 2, 4>(p, stream);
    case 96256: return launch_moe_wide<FORM, 2, 3, 4, 3>(p, stream);
    case 128128: return launch_moe_wide<FORM, 4, 2, 4, 4>(p, stream);
    case 128256: return launch_moe_wide<FORM, 4, 2, 8, 3>(p, stream);
    case 160128: return launch_moe_wide<FORM, 2, 5, 2, 4>(p, stream);
    case 160256: return launch_moe_wide<FORM, 2, 5, 4, 3>(p, stream);
    case 192128: return launch_moe_wide<FORM, 4, 3, 4, 4>(p, stream);
    case 192256: return launch_moe_wide<FORM, 4, 3, 8, 2>(p, stream);
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
