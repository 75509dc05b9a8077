// Kernels for mixers that carry a state of fixed size per request instead of a growing cache:
//
//   causal_conv            a short causal convolution per channel over the tokens of each sequence, whose last
//                          taps - 1 inputs are carried from step to step in the request's state slot;
//   conv_state_update      leaves those inputs for the next step;
//   rotary_to_float        rotary encoding of heads into float rows (what enters a recurrence stays in float);
//   linear_recurrence      S_t = a_t S_(t-1) + k_t (g_t v_t)^T,  y_t = S_t^T q_t + skip * v_t  per head, S [N, P] in float
//                          in the state slot: the state-space scan (k = B, q = C, v = x, a = exp(-exp(A_log) dt), g = dt,
//                          skip = D) and retention (a = the head's decay, g = 1, no skip) are both this recurrence;
//   gated_group_norm       the gate and the root-mean-square norm over groups of channels behind a recurrence, in
//                          either order;
//   mlstm_gates            log-domain input and forget gates of a matrix memory under a running maximum: the decays and
//                          input factors that make it the linear recurrence above;
//   mlstm_output           behind that recurrence: the division by the normaliser, the norm per head, the gate.
//
// A batch is token-major without padding: sequence s owns rows cu_seqlens[s] .. cu_seqlens[s + 1] - 1, its state
// sits in slot state_slots[s], and seq_starts[s] == 0 says that it starts now, from a zero state, whatever the slot
// held.  Sequences may have no rows at all.  All arithmetic is float; T is the storage type of rows.
#include "float_split.h"

#include <type_traits>

using namespace pllm;

__device__ __forceinline__ float load_as_f32(const void* p, int dtype, size_t i) {
  return dtype == PLLM_F32 ? reinterpret_cast<const float*>(p)[i] : __bfloat162float(reinterpret_cast<const bf16*>(p)[i]);
}
__device__ __forceinline__ float silu_f32(float z) { return z / (1.f + expf(-z)); }
// What a gate's raw value becomes behind a recurrence: z sigmoid(z), sigmoid(z), or 1 (no gate: nothing is read).
enum { kGateSilu = 0, kGateSigmoid = 1, kGateNone = 2 };
__device__ __forceinline__ float gate_f32(float z, int act) { return act == kGateSigmoid ? 1.f / (1.f + expf(-z)) : silu_f32(z); }

// ---------------------------------------------------------------------------------------------
constexpr int kMaxTaps = 16;      // most taps of a filter; filters of up to 8 taps take the smaller instance of the kernels
constexpr int kConvChunk = 64;     // tokens of one sequence that one workgroup walks: up to so many in one go (its state is then left by
constexpr int kConvShort = 16;     // the same kernel), else so many at a time, for workgroups enough to fill the GPU

// out[t, c] = act(bias[c] + sum_j w[c, j] * in[t - (taps - 1) + j, c]); the last column of w meets the current token;
// inputs before the sequence's first token of this step come from the state (or are zero for a sequence that starts).
// state: [slots][channels][taps - 1] floats, oldest input first.
template <typename T, int MAXT>
__global__ __launch_bounds__(256) void causal_conv_kernel(
    const T* __restrict__ in, int in_stride, const float* __restrict__ w, const float* __restrict__ bias,
    float* state, size_t slot_stride, const int* __restrict__ state_slots,
    const int* __restrict__ seq_starts, const int* __restrict__ cu_seqlens, T* __restrict__ out, int out_stride,
    int channels, int taps, int act, int leave_state, int chunk) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  const int seq = blockIdx.y;
  const int q_begin = cu_seqlens[seq], q_len = cu_seqlens[seq + 1] - q_begin;
  const int t0 = blockIdx.z * chunk;
  if (c >= channels || t0 >= q_len) return;
  const int t1 = t0 + chunk < q_len ? t0 + chunk : q_len;
  const bool carried = seq_starts[seq] > 0;
  float* st = state + (size_t)state_slots[seq] * slot_stride + (size_t)c * (taps - 1);
  float wj[MAXT], win[MAXT];
#pragma unroll
  for (int j = 0; j < MAXT; ++j) {
    wj[j] = j < taps ? w[(size_t)c * taps + j] : 0.f;
    win[j] = 0.f;
    if (j < taps - 1) {
      const int rel = t0 - (taps - 1) + j;      // token of this step (>= 0) or an input of earlier steps (< 0)
      if (rel >= 0) win[j] = to_f32(in[(size_t)(q_begin + rel) * in_stride + c]);
      else if (carried) win[j] = st[(taps - 1) + rel];
    }
  }
  const float b = bias ? bias[c] : 0.f;
  // Eight tokens' inputs are asked for at once: one wait for memory per eight tokens, not per token.
  constexpr int kAhead = 8;
  for (int tb = t0; tb < t1; tb += kAhead) {
    T fetched[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
      if (tb + u < t1) fetched[u] = in[(size_t)(q_begin + tb + u) * in_stride + c];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
    const int t = tb + u;
    if (t >= t1) break;
    const float cur = to_f32(fetched[u]);
    float acc = b;
#pragma unroll
    for (int j = 0; j < MAXT - 1; ++j)
      if (j < taps - 1) acc = fmaf(wj[j], win[j], acc);
#pragma unroll
    for (int j = 0; j < MAXT; ++j)
      if (j == taps - 1) acc = fmaf(wj[j], cur, acc);
#pragma unroll
    for (int j = 0; j < MAXT - 1; ++j) {
      if (j < taps - 2) win[j] = win[j + 1];
      else if (j == taps - 2) win[j] = cur;
    }
    out[(size_t)(q_begin + t) * out_stride + c] = from_f32<T>(act ? silu_f32(acc) : acc);
    }
  }
  // With one chunk per sequence this thread alone has read the channel's state, and what it holds now are the last
  // taps - 1 inputs: it leaves them itself (with several chunks another kernel does, after all of them have read).
  if (leave_state) {
#pragma unroll
    for (int j = 0; j < MAXT - 1; ++j)
      if (j < taps - 1) st[j] = win[j];
  }
}

template <typename T> struct alignas(4 * sizeof(T)) Quad { T v[4]; };

constexpr int kConvFours = 8;      // tokens of a workgroup of the kernel below

// The same with four taps and four neighbouring channels a thread, for portions in chunks.  The workgroups of a sequence's first chunk,
// which alone read the state, leave the new one.
// What bounds it: memory, and the exact SiLU's vector instructions (8 us of them at 2,048 tokens x 4,352 channels).  A thread's loads are
// 8 bytes (float rows 16) instead of 2, all of its tokens' under way at once, no tap is asked whether it is there, and no second kernel
// leaves the state.  us with what leaves the state, by channels and so: 2,048 tokens x 4,352 channels 28 and 15.4, 8 x 512 tokens
// 44 and 23.5.  Before its loads were asked for at once it took 17.4 there (16 tokens a workgroup 20.8), 1,178 x 2,048 13.1 and 8.8,
// 777 x 1,024 10.9 and 7.6; and the line was drawn: from 256 tokens on (100 tokens 11.0 and 11.2), and not beside more than a sixteenth as
// many sequences, where most workgroups have no tokens (65 tokens and 100 single ones 11.3 and 12.5).
template <typename T>
__global__ __launch_bounds__(256) void causal_conv4_kernel(
    const T* __restrict__ in, int in_stride, const float* __restrict__ w, const float* __restrict__ bias,
    float* state, size_t slot_stride, const int* __restrict__ state_slots,
    const int* __restrict__ seq_starts, const int* __restrict__ cu_seqlens, T* __restrict__ out, int out_stride, int channels, int act) {
  constexpr int kTaps = 4, V = 4;
  const int c = (blockIdx.x * blockDim.x + threadIdx.x) * V;
  const int seq = blockIdx.y, t0 = blockIdx.z * kConvFours;
  const int q_begin = cu_seqlens[seq], q_len = cu_seqlens[seq + 1] - q_begin, slot = state_slots[seq];
  const bool first = t0 == 0, carried = seq_starts[seq] > 0;
  if (c >= channels || (t0 >= q_len && !first)) return;
  float* st = state + (size_t)slot * slot_stride + (size_t)c * (kTaps - 1);
  if (q_len <= 0) {                                                    // no tokens: only an empty state is left
    if (!carried)
      for (int i = 0; i < V * (kTaps - 1); ++i) st[i] = 0.f;
    return;
  }
  const int count = min(kConvFours, q_len - t0);
  const T* rows = in + (size_t)(q_begin + t0) * in_stride + c;
  // Everything that memory holds for this thread is asked for before anything is used (rows that are not there as their neighbours): with the
  // inputs before the first, the weights and the bias each behind a wait of their own, 2,048 x 4,352 took 18.0 us and not 15.4.
  Quad<T> fetched[kConvFours], before[kTaps - 1];
#pragma unroll
  for (int u = 0; u < kConvFours; ++u) fetched[u] = *reinterpret_cast<const Quad<T>*>(rows + (size_t)min(u, count - 1) * in_stride);
#pragma unroll
  for (int j = 0; j < kTaps - 1; ++j) before[j] = *reinterpret_cast<const Quad<T>*>(rows + (first ? 0 : j - (kTaps - 1)) * (ptrdiff_t)in_stride);
  float wj[V][kTaps], win[V][kTaps - 1], b[V] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int v = 0; v < V; ++v)
#pragma unroll
    for (int j = 0; j < kTaps; ++j) wj[v][j] = w[(size_t)(c + v) * kTaps + j];
  if (bias) {
#pragma unroll
    for (int v = 0; v < V; ++v) b[v] = bias[c + v];
  }
  if (first) {
    float held[V][kTaps - 1];
    Quad<T> late[kTaps - 1];
#pragma unroll
    for (int v = 0; v < V; ++v)
#pragma unroll
      for (int j = 0; j < kTaps - 1; ++j) held[v][j] = st[v * (kTaps - 1) + j];
#pragma unroll
    for (int j = 0; j < kTaps - 1; ++j) late[j] = *reinterpret_cast<const Quad<T>*>(rows + (size_t)max(q_len - (kTaps - 1) + j, 0) * in_stride);
#pragma unroll
    for (int v = 0; v < V; ++v) {
#pragma unroll
      for (int j = 0; j < kTaps - 1; ++j) win[v][j] = carried ? held[v][j] : 0.f;
#pragma unroll
      for (int j = 0; j < kTaps - 1; ++j) {
        // (the last inputs of this step; with fewer than three the carried ones of one or two places on in front of them)
        const float kept = q_len == 1 ? win[v][j + 1 < kTaps - 1 ? j + 1 : 0] : win[v][j + 2 < kTaps - 1 ? j + 2 : 0];
        st[v * (kTaps - 1) + j] = q_len - (kTaps - 1) + j >= 0 ? to_f32(late[j].v[v]) : kept;
      }
    }
  } else {
#pragma unroll
    for (int v = 0; v < V; ++v)
#pragma unroll
      for (int j = 0; j < kTaps - 1; ++j) win[v][j] = to_f32(before[j].v[v]);
  }
#pragma unroll
  for (int u = 0; u < kConvFours; ++u) {
    Quad<T> o;
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const float cur = to_f32(fetched[u].v[v]);
      float acc = b[v];
#pragma unroll
      for (int j = 0; j < kTaps - 1; ++j) acc = fmaf(wj[v][j], win[v][j], acc);
      acc = fmaf(wj[v][kTaps - 1], cur, acc);
      win[v][0] = win[v][1];
      win[v][1] = win[v][2];
      win[v][2] = cur;
      o.v[v] = from_f32<T>(act ? silu_f32(acc) : acc);
    }
    if (u < count) *reinterpret_cast<Quad<T>*>(out + (size_t)(q_begin + t0 + u) * out_stride + c) = o;
  }
}

// state[k] <- the input at token q_len - (taps - 1) + k of this step, or what the state held for it.
template <typename T, int MAXT>
__global__ __launch_bounds__(256) void conv_state_update_kernel(
    const T* __restrict__ in, int in_stride, float* state, size_t slot_stride, const int* __restrict__ state_slots,
    const int* __restrict__ seq_starts, const int* __restrict__ cu_seqlens, int channels, int taps) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  const int seq = blockIdx.y;
  if (c >= channels) return;
  const int q_begin = cu_seqlens[seq], q_len = cu_seqlens[seq + 1] - q_begin;
  const bool carried = seq_starts[seq] > 0;
  float* st = state + (size_t)state_slots[seq] * slot_stride + (size_t)c * (taps - 1);
  float nv[MAXT];
#pragma unroll
  for (int k = 0; k < MAXT - 1; ++k) {
    nv[k] = 0.f;
    if (k < taps - 1) {
      const int rel = q_len - (taps - 1) + k;
      if (rel >= 0) nv[k] = to_f32(in[(size_t)(q_begin + rel) * in_stride + c]);
      else if (carried) nv[k] = st[q_len + k];
    }
  }
#pragma unroll
  for (int k = 0; k < MAXT - 1; ++k)
    if (k < taps - 1) st[k] = nv[k];
}

template <typename T, int MAXT>
static void launch_causal_conv(const void* in, int in_stride, const float* w, const float* bias, float* state, long slot_stride,
                               const int* state_slots, const int* seq_starts, const int* cu_seqlens, void* out, int out_stride,
                               int channels, int taps, int act, int num_seqs, int max_q_len, hipStream_t stream) {
  const int chunk = max_q_len <= kConvChunk ? kConvChunk : kConvShort;
  dim3 block(256), grid((channels + 255) / 256, num_seqs, (max_q_len + chunk - 1) / chunk);
  dim3 grid_state((channels + 255) / 256, num_seqs);
  const int fused = grid.z == 1 && taps > 1;
  const auto fours = [](const void* p, int stride) { return reinterpret_cast<uintptr_t>(p) % (4 * sizeof(T)) == 0 && stride % 4 == 0; };
  // (where each is ahead: above causal_conv4_kernel)
  const int fours_grid = (max_q_len + kConvFours - 1) / kConvFours;
  if (max_q_len >= 256 && num_seqs * 16 <= max_q_len && fours_grid <= 65535 && taps == 4 && channels % 4 == 0 && fours(in, in_stride) && fours(out, out_stride)) {
    hipLaunchKernelGGL(causal_conv4_kernel<T>, dim3((channels / 4 + 255) / 256, num_seqs, fours_grid), block, 0, stream, (const T*)in, in_stride, w, bias, state,
                       (size_t)slot_stride, state_slots, seq_starts, cu_seqlens, (T*)out, out_stride, channels, act);
  } else {
    hipLaunchKernelGGL((causal_conv_kernel<T, MAXT>), grid, block, 0, stream, (const T*)in, in_stride, w, bias, state,
                       (size_t)slot_stride, state_slots, seq_starts, cu_seqlens, (T*)out, out_stride, channels, taps, act, fused, chunk);
    if (taps > 1 && !fused)
      hipLaunchKernelGGL((conv_state_update_kernel<T, MAXT>), grid_state, block, 0, stream, (const T*)in, in_stride, state,
                         (size_t)slot_stride, state_slots, seq_starts, cu_seqlens, channels, taps);
  }
}

PLLM_API int pllm_causal_conv(int dtype, const void* in, int in_stride, const float* w, const float* bias, float* state,
                              long slot_stride, const int* state_slots, const int* seq_starts, const int* cu_seqlens,
                              void* out, int out_stride, int channels, int taps, int act, int num_seqs, int max_q_len,
                              hipStream_t stream) {
  if (num_seqs <= 0 || max_q_len <= 0 || channels <= 0) return 0;
  if (taps < 1 || taps > kMaxTaps) return -2;
#define PLLM_CONV(T, MAXT) launch_causal_conv<T, MAXT>(in, in_stride, w, bias, state, slot_stride, state_slots, seq_starts, cu_seqlens, \
                                                       out, out_stride, channels, taps, act, num_seqs, max_q_len, stream)
  if (dtype == PLLM_F32) { if (taps <= 8) PLLM_CONV(float, 8); else PLLM_CONV(float, kMaxTaps); }
  else { if (taps <= 8) PLLM_CONV(bf16, 8); else PLLM_CONV(bf16, kMaxTaps); }
#undef PLLM_CONV
  PLLM_RETURN_LAST_ERROR();
}

// ---------------------------------------------------------------------------------------------
// out[t, h, i] = float(rotated in[t, h, i]) * scale: the first rot_dims elements of each head turn by the angle of the
// token's position (tables cos/sin [positions, rot_dims / 2]); partners are (i, i + rot_dims / 2) or, interleaved,
// (2i, 2i + 1).  The result stays in float.
// blockIdx.y == 1: a second set of heads `second_at` columns further in the rows, into out + second_out, times scale2
// (the keys behind the queries).
template <typename T>
__global__ void rotary_to_float_kernel(const T* __restrict__ in, int in_stride, const int* __restrict__ positions,
                                       const float* __restrict__ cos_t, const float* __restrict__ sin_t, float* __restrict__ out,
                                       int heads, int head_dim, int rot_dims, int interleaved, float scale, int second_at,
                                       size_t second_out, float scale2) {
  const int tok = blockIdx.x;
  if (blockIdx.y == 1) { in += second_at; out += second_out; scale = scale2; }
  const int half = rot_dims / 2;
  const T* row = in + (size_t)tok * in_stride;
  const size_t table = (size_t)positions[tok] * half;
  for (int idx = threadIdx.x; idx < heads * head_dim; idx += blockDim.x) {
    const int h = idx / head_dim, i = idx % head_dim;
    const T* head = row + (size_t)h * head_dim;
    float val = to_f32(head[i]);
    if (i < rot_dims) {
      int pair, partner;
      bool upper;
      if (interleaved) { pair = i >> 1; upper = i & 1; partner = i ^ 1; }
      else { upper = i >= half; pair = upper ? i - half : i; partner = upper ? i - half : i + half; }
      const float other = to_f32(head[partner]);
      float lo, hi;
      rotate_pair(upper ? other : val, upper ? val : other, cos_t[table + pair], sin_t[table + pair], lo, hi);
      val = upper ? hi : lo;
    }
    out[(size_t)tok * heads * head_dim + idx] = val * scale;
  }
}

// The same in quads: a thread turns four pairs, or carries four elements behind the rotated ones over.
// What bounds it: memory (6 bytes an element from bfloat16: 5 TB/s at 2,048 tokens).  A thread of the kernel above asks for an element's
// partner again, for 4 bytes of a table and for 2 of a row at a time, behind two divisions.  us by elements and so, queries and keys of 8
// heads of 256: 2,048 tokens 20.3 and 10.0, 777 9.8 and 5.8, 8 or 1 as long as a launch takes; 16 of 64 in pairs of neighbours, 1,500 tokens
// 8.7 and 6.2; float rows of 8 of 128, half of it turned, 301 tokens 4.1 and 3.7.
template <typename T>
__global__ __launch_bounds__(256) void rotary_to_float_quads_kernel(const T* __restrict__ in, int in_stride, const int* __restrict__ positions,
                                                                    const float* __restrict__ cos_t, const float* __restrict__ sin_t,
                                                                    float* __restrict__ out, int heads, int head_dim, int rot_dims, int interleaved,
                                                                    float scale, int second_at, size_t second_out, float scale2) {
  const int tok = blockIdx.x;
  if (blockIdx.y == 1) { in += second_at; out += second_out; scale = scale2; }
  const int half = rot_dims / 2, turns = half / 4, items = turns + (head_dim - rot_dims) / 4;
  const T* row = in + (size_t)tok * in_stride;
  float* orow = out + (size_t)tok * heads * head_dim;
  const size_t table = (size_t)positions[tok] * half;
  for (int idx = threadIdx.x; idx < heads * items; idx += blockDim.x) {
    const int h = idx / items, r = idx - h * items, base = h * head_dim;
    if (r < turns) {
      const int at0 = base + (interleaved ? 8 * r : 4 * r), at1 = at0 + (interleaved ? 4 : half);
      const Quad<T> x0 = *reinterpret_cast<const Quad<T>*>(row + at0), x1 = *reinterpret_cast<const Quad<T>*>(row + at1);
      const Quad<float> c = *reinterpret_cast<const Quad<float>*>(cos_t + table + 4 * r), s = *reinterpret_cast<const Quad<float>*>(sin_t + table + 4 * r);
      float lo[4], hi[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const T even = i < 2 ? x0.v[2 * i & 3] : x1.v[2 * i & 3], odd = i < 2 ? x0.v[(2 * i & 3) + 1] : x1.v[(2 * i & 3) + 1];
        rotate_pair(to_f32(interleaved ? even : x0.v[i]), to_f32(interleaved ? odd : x1.v[i]), c.v[i], s.v[i], lo[i], hi[i]);
        lo[i] *= scale;
        hi[i] *= scale;
      }
      *reinterpret_cast<Quad<float>*>(orow + at0) = interleaved ? Quad<float>{lo[0], hi[0], lo[1], hi[1]} : Quad<float>{lo[0], lo[1], lo[2], lo[3]};
      *reinterpret_cast<Quad<float>*>(orow + at1) = interleaved ? Quad<float>{lo[2], hi[2], lo[3], hi[3]} : Quad<float>{hi[0], hi[1], hi[2], hi[3]};
    } else {
      const int at = base + rot_dims + 4 * (r - turns);
      const Quad<T> x = *reinterpret_cast<const Quad<T>*>(row + at);
      *reinterpret_cast<Quad<float>*>(orow + at) = Quad<float>{to_f32(x.v[0]) * scale, to_f32(x.v[1]) * scale, to_f32(x.v[2]) * scale, to_f32(x.v[3]) * scale};
    }
  }
}

PLLM_API int pllm_rotary_to_float(int dtype, const void* in, int in_stride, const int* positions, const float* cos_t,
                                  const float* sin_t, float* out, int num_tokens, int heads, int head_dim, int rot_dims,
                                  int interleaved, float scale, int sets, int second_at, long second_out, float scale2,
                                  hipStream_t stream) {
  if (num_tokens <= 0) return 0;
  if (rot_dims < 0 || rot_dims > head_dim || rot_dims % 2 || sets < 1 || sets > 2) return -2;
  dim3 grid(num_tokens, sets), block(256);
  // Quads where everything that they load and store lies on their boundaries (figures: above the kernel).
  const uintptr_t size = dtype == PLLM_F32 ? 4 : 2;
  const bool quads = rot_dims % 8 == 0 && head_dim % 4 == 0 && in_stride % 4 == 0 && second_at % 4 == 0 && second_out % 4 == 0 &&
                     (uintptr_t)in % (4 * size) == 0 && ((uintptr_t)out | (uintptr_t)cos_t | (uintptr_t)sin_t) % 16 == 0;
#define PLLM_ROTARY(KERNEL, T) hipLaunchKernelGGL(KERNEL<T>, grid, block, 0, stream, (const T*)in, in_stride, positions, cos_t, sin_t, \
                                                  out, heads, head_dim, rot_dims, interleaved, scale, second_at, (size_t)second_out, scale2)
  if (dtype == PLLM_F32) { if (quads) PLLM_ROTARY(rotary_to_float_quads_kernel, float); else PLLM_ROTARY(rotary_to_float_kernel, float); }
  else { if (quads) PLLM_ROTARY(rotary_to_float_quads_kernel, bf16); else PLLM_ROTARY(rotary_to_float_kernel, bf16); }
#undef PLLM_ROTARY
  PLLM_RETURN_LAST_ERROR();
}

// ---------------------------------------------------------------------------------------------
struct RecurrenceArgs {
  const void* q; const void* k;        // [T, key_heads, N], element type qk_dtype, row stride qk_stride (elements)
  const void* v;                       // [T, heads, P], element type v_dtype, row stride v_stride
  const float* decay;                  // a_t per head: decay[t * decay_stride + h] (decay_stride 0: one number per head)
  const float* row_decay;              // or a decay per row of S: row_decay[t * row_decay_stride + h * N + n] (then `decay` is null and
                                       // S_t = diag(row_decay_t) S_(t-1) + k_t (g_t v_t)^T); not together with raw step sizes
  int row_decay_stride;
  const float* vscale;                 // g_t per head [T, heads], or null for 1
  // or both from raw step sizes [T, heads] (element type raw_dtype, row stride raw_stride):
  //   g_t = softplus(raw + raw_bias[h]) (no clamp),  a_t = exp(-exp(a_log[h]) * g_t)
  const void* raw; const float* raw_bias; const float* a_log;
  int raw_dtype, raw_stride;
  const float* skip;                   // [heads] or null
  float* state;                        // slot s, head h: state + s * slot_stride + h * N * P, as [N][P]
  const int* state_slots; const int* seq_starts; const int* cu_seqlens;
  float* out;                          // [T, heads * P]
  long slot_stride;
  int qk_dtype, qk_stride, v_dtype, v_stride, decay_stride;
  int heads, key_heads, N, P, pblocks;
  int ld;                              // elements of a row of S in the state and of a head in the output rows: P, or P + 1 when a
                                       // normaliser n_t = a_t n_(t-1) + g_t k_t stands behind the P columns (n as the last column of
                                       // S, n_t . q_t as the last element of the head's output)
};

// One workgroup per (sequence or chunk, head, block of 64 value channels); lane = value channel, so a token's update
// needs no exchange between lanes.  Wave w holds rows w * NR .. w * NR + NR - 1 of S in registers; with several waves
// their partial outputs are added through LDS in wave order.  A token's k and q are fetched by one lane each and read
// out lane by lane.
//
// Three forms (MODE):
//   kWhole       a sequence's tokens of this step one after the other, from the slot's state to the slot's state: steps
//                of single tokens and short portions;
//   kChunkState  long portions, first pass: the tokens of one chunk from a zero state, no outputs; leaves the chunk's
//                own contribution S_loc and the product of its decays in the workspace;
//   kChunkOut    third pass: a chunk's tokens from the state the sequence had when the chunk began (which the second
//                pass, recurrence_carry_kernel, has put where S_loc was), with outputs, no state written.
// With chunks, a long prompt's tokens are spread over the whole GPU instead of one workgroup per head; the additions
// into S associate differently than token by token, so results differ from the whole form by float rounding.
enum { kWhole = 0, kChunkState = 1, kChunkOut = 2 };

struct ChunkArgs {
  float* ws_state;      // [chunks][heads][N][P]
  float* ws_decay;      // [chunks][heads], or [chunks][heads][N] with a decay per row
  int chunk;            // tokens per chunk
  int num_seqs;
};

// Chunk j of the batch: sequences in order, each with ceil(q_len / chunk) chunks.  False when j is past the last one.
__device__ __forceinline__ bool find_chunk(const int* __restrict__ cu_seqlens, int num_seqs, int chunk, int j, int& seq, int& local) {
  int base = 0;
  for (int s = 0; s < num_seqs; ++s) {
    const int c = (cu_seqlens[s + 1] - cu_seqlens[s] + chunk - 1) / chunk;
    if (j < base + c) { seq = s; local = j - base; return true; }
    base += c;
  }
  return false;
}

template <int NR, int MAX_THREADS, int MODE>
__global__ __launch_bounds__(MAX_THREADS) void linear_recurrence_kernel(RecurrenceArgs a, ChunkArgs ca) {
  __shared__ float part[2][MAX_THREADS / 64][64];
  __shared__ float part_n[2][MAX_THREADS / 64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const int head = blockIdx.x / a.pblocks, pb = blockIdx.x % a.pblocks;
  const int p = pb * 64 + lane;
  const bool p_ok = p < a.P;
  int seq = blockIdx.y, local = 0;
  if (MODE != kWhole && !find_chunk(a.cu_seqlens, ca.num_seqs, ca.chunk, blockIdx.y, seq, local)) return;
  const int q_begin = a.cu_seqlens[seq], q_len = a.cu_seqlens[seq + 1] - q_begin;
  if (q_len <= 0) return;
  const int t_first = MODE == kWhole ? 0 : local * ca.chunk;
  const int t_last = MODE == kWhole ? q_len : (t_first + ca.chunk < q_len ? t_first + ca.chunk : q_len);
  const int kh = head / (a.heads / a.key_heads);
  const int n0 = wv * NR;
  const bool carried = a.seq_starts[seq] > 0;
  const int ld = a.ld;
  float* st = MODE == kWhole ? a.state + (size_t)a.state_slots[seq] * a.slot_stride + (size_t)head * a.N * ld
                             : ca.ws_state + ((size_t)blockIdx.y * a.heads + head) * a.N * ld;
  const bool from_state = MODE != kChunkState && (MODE == kChunkOut || carried);
  float S[NR];
#pragma unroll
  for (int i = 0; i < NR; ++i) S[i] = (from_state && p_ok && n0 + i < a.N) ? st[(size_t)(n0 + i) * ld + p] : 0.f;
  const float skip = a.skip ? a.skip[head] : 0.f;
  const float rate = a.raw ? expf(a.a_log[head]) : 0.f, raw_bias = a.raw ? a.raw_bias[head] : 0.f;
  const bool mine = lane < NR && n0 + lane < a.N;
  // The normaliser, where there is one: lane l of wave w holds n[w * NR + l], the row whose k and q it fetches anyway, so its
  // update is one multiply-add a token and n . q one sum over the wavefront; the head's first block of columns keeps it.
  const bool with_n = ld > a.P && pb == 0;
  float nl = (with_n && from_state && mine) ? st[(size_t)(n0 + lane) * ld + a.P] : 0.f;
  float decays = 1.f;
  // What a token needs from memory is asked for one token ahead, so that it travels while the token before is computed.
  struct Fetched { float k, q, x, a, g, d; };
  const bool by_row = a.row_decay != nullptr;
  float decays_l = 1.f;                                      // with a decay per row: the product for row n0 + lane
  auto fetch = [&](int t) {
    Fetched f;
    const size_t row = (size_t)(q_begin + t);
    const size_t qk_at = row * a.qk_stride + (size_t)kh * a.N + n0 + lane;
    f.k = mine ? load_as_f32(a.k, a.qk_dtype, qk_at) : 0.f;
    f.q = (MODE != kChunkState && mine) ? load_as_f32(a.q, a.qk_dtype, qk_at) : 0.f;
    f.x = p_ok ? load_as_f32(a.v, a.v_dtype, row * a.v_stride + (size_t)head * a.P + p) : 0.f;
    f.d = 1.f;
    if (by_row) {
      f.d = mine ? a.row_decay[row * a.row_decay_stride + (size_t)head * a.N + n0 + lane] : 1.f;
      f.a = 1.f;
      f.g = a.vscale ? a.vscale[row * a.heads + head] : 1.f;
    } else if (a.raw) {
      f.a = load_as_f32(a.raw, a.raw_dtype, row * a.raw_stride + head);
      f.g = 0.f;
    } else {
      f.a = a.decay[row * a.decay_stride + head];
      f.g = a.vscale ? a.vscale[row * a.heads + head] : 1.f;
    }
    return f;
  };
  // The state pass walks its chunk from the last token to the first: the chunk's own contribution is the sum over its
  // tokens of k_t (g_t v_t)^T times the decays of the tokens behind t, and that product is at hand when t is reached
  // from behind: one multiply-add per state row and token, no decay of the rows.
  Fetched next = fetch(MODE == kChunkState ? t_last - 1 : t_first);
  for (int n = t_first; n < t_last; ++n) {
    const int t = MODE == kChunkState ? t_last - 1 - (n - t_first) : n;
    const Fetched cur = next;
    if (n + 1 < t_last) next = fetch(MODE == kChunkState ? t - 1 : t + 1);
    const size_t row = (size_t)(q_begin + t);
    const float k_l = cur.k, q_l = cur.q, x = cur.x;
    float dec, xg, g;
    if (a.raw) {
      const float z = cur.a + raw_bias;
      const float step = z > 20.f ? z : log1pf(expf(z));
      dec = expf(-rate * step);
      g = step;
    } else {
      dec = cur.a;
      g = cur.g;
    }
    xg = x * g;
    if (by_row) {
      const float d_l = cur.d;
      if (MODE == kChunkState) {
        const float kw = k_l * decays_l;                  // decays_l: of the tokens behind t in the chunk, for this lane's row
#pragma unroll
        for (int i = 0; i < NR; ++i) S[i] = fmaf(row_lane(kw, i), xg, S[i]);
        if (with_n) nl = fmaf(kw, g, nl);
        decays_l *= d_l;
        continue;
      }
      float nq = 0.f;
      if (with_n) {
        nl = fmaf(k_l, g, d_l * nl);
        nq = wave_sum(nl * q_l);
      }
      float y[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        const float kk = row_lane(k_l, i), qq = row_lane(q_l, i), dd = row_lane(d_l, i);
        S[i] = fmaf(kk, xg, dd * S[i]);
        y[i & 3] = fmaf(S[i], qq, y[i & 3]);
      }
      float total = (y[0] + y[1]) + (y[2] + y[3]);
      if (waves > 1) {
        part[t & 1][wv][lane] = total;
        if (with_n && lane == 0) part_n[t & 1][wv] = nq;
        __syncthreads();
        if (wv == 0) {
          total = part[t & 1][0][lane];
          for (int w = 1; w < waves; ++w) total += part[t & 1][w][lane];
          if (with_n) {
            nq = part_n[t & 1][0];
            for (int w = 1; w < waves; ++w) nq += part_n[t & 1][w];
          }
        }
      }
      if (wv == 0 && p_ok) a.out[row * (size_t)(a.heads * ld) + (size_t)head * ld + p] = fmaf(skip, x, total);
      if (wv == 0 && with_n && lane == 0) a.out[row * (size_t)(a.heads * ld) + (size_t)head * ld + a.P] = nq;
      continue;
    }
    if (MODE == kChunkState) {
      const float xw = xg * decays;                       // decays: of the tokens behind t in the chunk
#pragma unroll
      for (int i = 0; i < NR; ++i) S[i] = fmaf(row_lane(k_l, i), xw, S[i]);
      if (with_n) nl = fmaf(k_l, g * decays, nl);
      decays *= dec;
      continue;
    }
    float nq = 0.f;
    if (with_n) {
      nl = fmaf(k_l, g, dec * nl);
      nq = wave_sum(nl * q_l);
    }
    float y[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const float kk = row_lane(k_l, i), qq = row_lane(q_l, i);
      S[i] = fmaf(kk, xg, dec * S[i]);
      y[i & 3] = fmaf(S[i], qq, y[i & 3]);
    }
    float total = (y[0] + y[1]) + (y[2] + y[3]);
    if (waves > 1) {
      part[t & 1][wv][lane] = total;
      if (with_n && lane == 0) part_n[t & 1][wv] = nq;
      __syncthreads();
      if (wv == 0) {
        total = part[t & 1][0][lane];
        for (int w = 1; w < waves; ++w) total += part[t & 1][w][lane];
        if (with_n) {
          nq = part_n[t & 1][0];
          for (int w = 1; w < waves; ++w) nq += part_n[t & 1][w];
        }
      }
    }
    if (wv == 0 && p_ok) a.out[row * (size_t)(a.heads * ld) + (size_t)head * ld + p] = fmaf(skip, x, total);
    if (wv == 0 && with_n && lane == 0) a.out[row * (size_t)(a.heads * ld) + (size_t)head * ld + a.P] = nq;
  }
  if (MODE == kChunkOut) return;
  if (p_ok) {
#pragma unroll
    for (int i = 0; i < NR; ++i)
      if (n0 + i < a.N) st[(size_t)(n0 + i) * ld + p] = S[i];
  }
  if (with_n && mine) st[(size_t)(n0 + lane) * ld + a.P] = nl;
  if (MODE == kChunkState && by_row) {
    if (pb == 0 && mine) ca.ws_decay[((size_t)blockIdx.y * a.heads + head) * a.N + n0 + lane] = decays_l;
  } else if (MODE == kChunkState && threadIdx.x == 0 && pb == 0) ca.ws_decay[(size_t)blockIdx.y * a.heads + head] = decays;
}

// Second pass: per sequence and state element, chunk after chunk:  ws[c] <- the state before chunk c,
// S <- decays[c] * S + S_loc[c];  the state after the last chunk goes to the slot.
__global__ __launch_bounds__(256) void recurrence_carry_kernel(RecurrenceArgs a, ChunkArgs ca) {
  const size_t per_head = (size_t)a.N * a.ld, per_seq = per_head * a.heads;
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int seq = blockIdx.y;
  if (idx >= per_seq) return;
  const int q_len = a.cu_seqlens[seq + 1] - a.cu_seqlens[seq];
  if (q_len <= 0) return;
  int base = 0;
  for (int s = 0; s < seq; ++s) base += (a.cu_seqlens[s + 1] - a.cu_seqlens[s] + ca.chunk - 1) / ca.chunk;
  const int chunks = (q_len + ca.chunk - 1) / ca.chunk;
  const int head = (int)(idx / per_head);
  const size_t decay_at = a.row_decay ? (size_t)head * a.N + (idx - (size_t)head * per_head) / a.ld : (size_t)head;
  const size_t decay_ld = a.row_decay ? (size_t)a.heads * a.N : (size_t)a.heads;
  float* slot = a.state + (size_t)a.state_slots[seq] * a.slot_stride + idx;
  float S = a.seq_starts[seq] > 0 ? *slot : 0.f;
  for (int c = 0; c < chunks; ++c) {
    float* w = ca.ws_state + (size_t)(base + c) * per_seq + idx;
    const float loc = *w;
    *w = S;
    S = fmaf(ca.ws_decay[(size_t)(base + c) * decay_ld + decay_at], S, loc);
  }
  *slot = S;
}

// (Chunks come here only for what the matrix forms below do not take: more than 256 rows, 128 with a decay per row, and rows 2^22 elements apart.)
template <int MODE>
static void launch_recurrence(const RecurrenceArgs& a, const ChunkArgs& ca, dim3 grid, int waves, int need, hipStream_t stream) {
  dim3 block(64 * waves);
  if (waves > 4) {
    hipLaunchKernelGGL((linear_recurrence_kernel<64, 1024, MODE>), grid, block, 0, stream, a, ca);
    return;
  }
  if constexpr (MODE == kWhole) {
    if (need <= 8) {
      hipLaunchKernelGGL((linear_recurrence_kernel<8, 256, MODE>), grid, block, 0, stream, a, ca);
      return;
    }
    if (need <= 16) {
      hipLaunchKernelGGL((linear_recurrence_kernel<16, 256, MODE>), grid, block, 0, stream, a, ca);
      return;
    }
    if (need <= 32) {
      hipLaunchKernelGGL((linear_recurrence_kernel<32, 256, MODE>), grid, block, 0, stream, a, ca);
      return;
    }
  }
  hipLaunchKernelGGL((linear_recurrence_kernel<64, 256, MODE>), grid, block, 0, stream, a, ca);
}

// ---------------------------------------------------------------------------------------------
// The first and the third pass with a decay per row as matrix products in float (v_mfma_f32_16x16x4_f32), for heads of up to 128 rows: a
// workgroup walks its chunk in pieces of 32 tokens.  With D[t, j] the products (one per row) of the decays of tokens j + 1 .. t of a
// piece, G_t those of its tokens up to t and S the state in front of it,
//   Y = (G Q) S + M V + skip V,   M[t, j] = g_j (q_t . D[t, j] k_j) for j <= t,
//   S <- G_32 S + (D[32, j] K)^T (g_j V)
// (every product of decays is built by multiplication, none from a difference of logarithms: as many roundings as token by
// token).  The decays stand inside the sums over the rows: there G Q and K^T carry them element by element; M's tile of
// late queries and early keys takes both from the tiles' border (no factor is above 1), and its two tiles on the diagonal are
// summed by vector instructions, a thread walking the queries behind one key with the key's rows times their decays at hand.
//
// A wavefront owns 16 columns of S and all of its rows in registers.  A result's lane (g, c) = (lane >> 4, lane & 15) holds
// rows 4 g .. 4 g + 3 of column c, and such a fragment of S is the operand of Y^T = S^T Q^T as it stands; so is one of M.
// K and V lie in LDS by rows of S and columns (tokens in fours, in an order that spreads the banks).  The next piece's rows
// travel while this one is worked off.
//
// What bounds it: the float matrix cores (a third to half busy) beside a piece's barriers and its way through LDS.  A prompt
// of 2,048 tokens, one layer, states + carry + outputs, 16 heads of 128 x 128: 232 us token by token in chunks of 64 -> 131 us.  Errors
// against 64 bits over 1 to 2,048 tokens: outputs 2.6e-8 to 1.5e-6 as before or below, the last states below (1.1e-7 against
// 2.0e-7, 2.1e-6 against 6.3e-6).
constexpr int kPiece = 32, kPieceLd = kPiece + 4;

typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma16(const f32x4 a, const f32x4 b, f32x4 acc) {
#pragma unroll
  for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], acc, 0, 0, 0);
  return acc;
}
// The products of sixteen rows of one operand and sixteen of the other over 16 NT elements, in four sums: a chain of
// roundings as short as the token-by-token kernel's.
template <int NT>
__device__ __forceinline__ f32x4 dot_rows(const float* a, const float* b) {
  f32x4 part[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) part[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < NT; ++i) part[i & 3] = mfma16(*reinterpret_cast<const f32x4*>(a + 16 * i), *reinterpret_cast<const f32x4*>(b + 16 * i), part[i & 3]);
  return (part[0] + part[1]) + (part[2] + part[3]);
}
// Where four tokens 4 f .. 4 f + 3 of row n stand in an array of rows over the tokens of a piece.
__device__ __forceinline__ int token_quad(int n, int f) { return n * kPiece + ((f ^ n ^ (n >> 3)) & 7) * 4; }
__device__ __forceinline__ f32x4 lds_quad(const float* p) { return *reinterpret_cast<const f32x4*>(p); }

// Elements n .. n + 3 of a row that holds `count`, zeros past it.  vec: they can be read at once and never straddle the end.
__device__ __forceinline__ f32x4 row_quad(const void* base, int dtype, size_t at, int n, int count, bool vec) {
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  if (n >= count) return v;
  if (!vec) {
    v[0] = load_as_f32(base, dtype, at);
    if (n + 1 < count) v[1] = load_as_f32(base, dtype, at + 1);
    if (n + 2 < count) v[2] = load_as_f32(base, dtype, at + 2);
    if (n + 3 < count) v[3] = load_as_f32(base, dtype, at + 3);
    return v;
  }
  if (dtype == PLLM_F32) return *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(base) + at);
  const uint2 w = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint16_t*>(base) + at);
  v[0] = __uint_as_float(w.x << 16); v[1] = __uint_as_float(w.x & 0xffff0000u);
  v[2] = __uint_as_float(w.y << 16); v[3] = __uint_as_float(w.y & 0xffff0000u);
  return v;
}

constexpr int kVecRows = 1, kVecValues = 2, kVecOut = 4, kVecDecay = 8;

// Floats of LDS, in the order the kernel lays them out.
template <int NT, int WAVES, int MODE> constexpr int piece_lds_floats() {
  constexpr int NP = 16 * NT, rows = kPiece * (NP + 4), half = (kPiece / 2) * (NP + 4);
  int n = NP * kPiece + 16 * WAVES * kPiece;                                     // K^T, V^T
  if (MODE != kChunkState) n += 2 * rows + kPiece * kPieceLd;                      // Q, K, M
  n += rows + NP + kPiece + (MODE != kChunkState ? 2 * half : rows);              // decays, G_32, g; late queries, early keys (first pass: K)
  return n;
}

template <int NT, int WAVES, int MODE>
__global__ __launch_bounds__(64 * WAVES, 2) void recurrence_piece_kernel(RecurrenceArgs a, ChunkArgs ca, int vec) {
  constexpr int NP = 16 * NT, LD = NP + 4, kThreads = 64 * WAVES, kQuads = (kPiece * NP / 4 + kThreads - 1) / kThreads;
  constexpr bool kOut = MODE != kChunkState;                           // (kWhole: a sequence from the slot's state to the slot's state)
  extern __shared__ __attribute__((aligned(16))) unsigned char piece_lds[];
  float* KT = reinterpret_cast<float*>(piece_lds);                     // [NP][32]
  float* VT = KT + NP * kPiece;                                        // [16 WAVES][32]
  float* Q = VT + 16 * WAVES * kPiece;                                 // [32][LD]  q, then G q
  float* K = kOut ? Q + kPiece * LD : Q;                               // [32][LD]
  float* M = K + kPiece * LD;                                          // [32][kPieceLd]
  float* DR = kOut ? M + kPiece * kPieceLd : M;                        // [32][LD] decays
  float* gC = DR + kPiece * LD;                                        // [NP]
  float* gs = gC + NP;                                                 // [32] g
  float* Q2 = gs + kPiece;                                             // [16][LD] late queries, decayed from token 16 on
  float* K2 = Q2 + (kPiece / 2) * LD;                                  // [16][LD] early keys, decayed up to token 15
  const int tid = threadIdx.x, lane = tid & 63, c16 = lane & 15, quad = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int head = blockIdx.x / a.pblocks, pb = blockIdx.x % a.pblocks;
  int seq = blockIdx.y, local = 0;
  if (MODE != kWhole && !find_chunk(a.cu_seqlens, ca.num_seqs, ca.chunk, blockIdx.y, seq, local)) return;
  const int q_begin = a.cu_seqlens[seq], q_len = a.cu_seqlens[seq + 1] - q_begin;
  if (q_len <= 0) return;
  const int t_first = MODE == kWhole ? 0 : local * ca.chunk, t_last = MODE == kWhole ? q_len : min(t_first + ca.chunk, q_len);
  const int kh = head / (a.heads / a.key_heads), ld = a.ld, p0 = pb * 16 * WAVES;
  const int p = p0 + 16 * wave + c16;                                  // this lane's column of S
  float* st = MODE == kWhole ? a.state + (size_t)a.state_slots[seq] * a.slot_stride + (size_t)head * a.N * ld
                             : ca.ws_state + ((size_t)blockIdx.y * a.heads + head) * a.N * ld;
  const bool from_state = MODE == kChunkOut || (MODE == kWhole && a.seq_starts[seq] > 0);
  const bool live = p0 + 16 * wave < ld;                               // (the wavefront has columns)

  f32x4 S[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = 16 * i + 4 * quad + r;
      S[i][r] = from_state && p < ld && n < a.N ? st[(size_t)n * ld + p] : 0.f;
    }
  const float skip = a.skip ? a.skip[head] : 0.f;

  f32x4 rq[kOut ? kQuads : 1], rk[kQuads], rd[kQuads], rv[2];
  float rg = 1.f;                                                      // g of token tid
  auto fetch = [&](int t0) {
#pragma unroll
    for (int e = 0; e < kQuads; ++e) {
      const int at = tid + e * kThreads, t = at / (NP / 4), n = at % (NP / 4) * 4;
      const bool in = t < kPiece && t0 + t < t_last;
      const size_t row = (size_t)(q_begin + (in ? t0 + t : t_first));
      const int most = in ? a.N : 0;
      rk[e] = row_quad(a.k, a.qk_dtype, row * a.qk_stride + (size_t)kh * a.N + n, n, most, vec & kVecRows);
      if (kOut) rq[e] = row_quad(a.q, a.qk_dtype, row * a.qk_stride + (size_t)kh * a.N + n, n, most, vec & kVecRows);
      rd[e] = row_quad(a.row_decay, PLLM_F32, row * a.row_decay_stride + (size_t)head * a.N + n, n, most, vec & kVecDecay);
      if (!in) rd[e] = f32x4{1.f, 1.f, 1.f, 1.f};
    }
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int at = tid + e * kThreads, t = at / (4 * WAVES), col = p0 + at % (4 * WAVES) * 4;
      const bool in = t0 + t < t_last;
      const size_t row = (size_t)(q_begin + (in ? t0 + t : t_first));
      rv[e] = row_quad(a.v, a.v_dtype, row * a.v_stride + (size_t)head * a.P + col, col, in ? a.P : 0, vec & kVecValues);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (in && ld > a.P && col + i == a.P) rv[e][i] = 1.f;          // the normaliser's column
    }
    if (tid < kPiece) rg = a.vscale && t0 + tid < t_last ? a.vscale[(size_t)(q_begin + t0 + tid) * a.heads + head] : 1.f;
  };
  fetch(t_first);
  float total = 1.f;                                                   // first pass: the product of the chunk's decays

  for (int t0 = t_first; t0 < t_last; t0 += kPiece) {
    const bool last = t0 + kPiece >= t_last;
    __syncthreads();                                                   // the piece before is done with LDS
    bool odd = false;                                                  // a value that is no number (see below)
#pragma unroll
    for (int e = 0; e < kQuads; ++e) {
      const int at = tid + e * kThreads, t = at / (NP / 4), n = at % (NP / 4) * 4;
      if (kPiece * NP / 4 % kThreads && t >= kPiece) break;
      if (kOut) *reinterpret_cast<f32x4*>(Q + t * LD + n) = rq[e];
      *reinterpret_cast<f32x4*>(K + t * LD + n) = rk[e];
      *reinterpret_cast<f32x4*>(DR + t * LD + n) = rd[e];
    }
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int at = tid + e * kThreads, t = at / (4 * WAVES), col = at % (4 * WAVES) * 4;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float x = rv[e][i];
        VT[token_quad(col + i, t >> 2) + (t & 3)] = x;
        odd = odd || !(fabsf(x) < INFINITY);
      }
    }
    if (tid < kPiece) gs[tid] = rg;
    odd = kOut && __syncthreads_or(odd);
    if (!kOut) __syncthreads();
    if (!last) fetch(t0 + kPiece);

    // Four walks along the tokens, a row a thread: late queries and the piece's product forward, all keys and early keys backward.
    for (int who = tid; who < 4 * NP; who += kThreads) {
      const int n = who % NP, walk = who / NP;
      if (walk == 0) {
        if (kOut) {
          float from16 = 1.f;
#pragma unroll 4
          for (int t = kPiece / 2; t < kPiece; ++t) {
            from16 *= DR[t * LD + n];
            Q2[(t - kPiece / 2) * LD + n] = Q[t * LD + n] * from16;
          }
        }
      } else if (walk == 1) {
        float all = 1.f;
#pragma unroll 4
        for (int t = 0; t < kPiece; ++t) all *= DR[t * LD + n];
        gC[n] = all;
      } else if (walk == 2) {
        float behind = 1.f;
#pragma unroll 4
        for (int t = kPiece - 1; t >= 0; --t) {
          KT[token_quad(n, t >> 2) + (t & 3)] = K[t * LD + n] * behind * gs[t];
          behind *= DR[t * LD + n];
        }
      } else if (kOut) {
        float to15 = 1.f;
#pragma unroll 4
        for (int t = kPiece / 2 - 1; t >= 0; --t) {
          K2[t * LD + n] = K[t * LD + n] * to15;
          to15 *= DR[t * LD + n];
        }
      }
    }
    if constexpr (kOut) {
      // The tiles of M on the diagonal: sixteen lanes share a key, NT of its rows each, added in their order and then over the lanes.
      // What bounds it is LDS: so every sixteen lanes take two keys, a token's decays and queries read for both, and nothing stands
      // behind a condition, so that the reads of the tokens to come are under way (16 heads
      // of 128 x 128, 777 tokens in pieces 441 -> 289 us with the walks above, in chunks 66.5 -> 55.5; 64 of 64 x 64 333 -> 224 and 94 -> 73).
      for (int eight = wave; eight < 4; eight += WAVES) {
        const int first = (eight >> 1) * 16, j0 = first + (eight & 1) * 8 + quad, n = c16 * NT;      // keys j0 and j0 + 4
        float w[2][NT];
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
          for (int i = 0; i < NT; ++i) w[k][i] = K[(j0 + 4 * k) * LD + n + i];
        const float g = gs[j0 + 4 * (c16 & 1)];
#pragma unroll 4
        for (int t = first; t < first + 16; ++t) {
          float d[NT], q[NT], dot[2];
#pragma unroll
          for (int i = 0; i < NT; ++i) { d[i] = DR[t * LD + n + i]; q[i] = Q[t * LD + n + i]; }
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            const int j = j0 + 4 * k;
            dot[k] = 0.f;
#pragma unroll
            for (int i = 0; i < NT; ++i) {
              w[k][i] = t > j ? w[k][i] * d[i] : w[k][i];
              dot[k] = fmaf(w[k][i], q[i], dot[k]);
            }
            dot[k] += dpp_move<kDppSwap1>(dot[k]);
            dot[k] += dpp_move<kDppSwap2>(dot[k]);
            dot[k] += dpp_move<kDppHalfMirror>(dot[k]);
            dot[k] += dpp_move<kDppMirror>(dot[k]);
          }
          // (a key behind the token: zero, whatever its gain is)
          if (c16 < 2) M[t * kPieceLd + j0 + 4 * c16] = t >= j0 + 4 * c16 ? (c16 ? dot[1] : dot[0]) * g : 0.f;
        }
      }
      __syncthreads();
      for (int n = tid; n < NP; n += kThreads) {                     // (the diagonal is done with the plain queries)
        float all = 1.f;
#pragma unroll 4
        for (int t = 0; t < kPiece; ++t) {
          all *= DR[t * LD + n];
          Q[t * LD + n] *= all;
        }
      }
      if (wave == WAVES - 1) {                                       // late queries, early keys
        const f32x4 m = dot_rows<NT>(K2 + c16 * LD + 4 * quad, Q2 + c16 * LD + 4 * quad);
        *reinterpret_cast<f32x4*>(M + (16 + c16) * kPieceLd + 4 * quad) = m * lds_quad(gs + 4 * quad);
      }
    }
    __syncthreads();
    f32x4 v[2], y[2], carried[2];
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      v[f] = lds_quad(VT + token_quad(16 * wave + c16, 4 * f + quad));
      y[f] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    if (kOut && live) {
      f32x4 part[4][2];                                                // (four sums, as in dot_rows)
#pragma unroll
      for (int f = 0; f < 2; ++f) part[0][f] = part[1][f] = part[2][f] = part[3][f] = y[f];
#pragma unroll
      for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int f = 0; f < 2; ++f) part[i & 3][f] = mfma16(S[i], lds_quad(Q + (16 * f + c16) * LD + 16 * i + 4 * quad), part[i & 3][f]);
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        carried[f] = (part[0][f] + part[1][f]) + (part[2][f] + part[3][f]);
      }
    }
    if ((MODE != kChunkOut || !last) && live) {
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        S[i] *= lds_quad(gC + 16 * i + 4 * quad);
#pragma unroll
        for (int f = 0; f < 2; ++f) S[i] = mfma16(lds_quad(KT + token_quad(16 * i + c16, 4 * f + quad)), v[f], S[i]);
      }
    }
    if (!kOut) {
      if (pb == 0 && tid < a.N) {
        total *= gC[tid];
        if (last) ca.ws_decay[((size_t)blockIdx.y * a.heads + head) * a.N + tid] = total;
      }
    }
    if constexpr (kOut) {
      if (live) {
        // (A weight of zero must not meet a value that is no number: such a value reaches its own token and later ones only.)
        f32x4 fine[2] = {v[0], v[1]};
        if (odd) {
#pragma unroll
          for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (!(fabsf(fine[f][r]) < INFINITY)) fine[f][r] = 0.f;
#pragma unroll 1
          for (int j = 0; j < kPiece; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float x = VT[token_quad(16 * wave + 4 * quad + r, j >> 2) + (j & 3)];
              if (fabsf(x) < INFINITY) continue;
#pragma unroll
              for (int f = 0; f < 2; ++f)
                if (j <= 16 * f + c16) y[f][r] = fmaf(M[(16 * f + c16) * kPieceLd + j], x, y[f][r]);
            }
        }
        y[0] = mfma16(fine[0], lds_quad(M + c16 * kPieceLd + 4 * quad), y[0]);
        y[1] = mfma16(fine[0], lds_quad(M + (16 + c16) * kPieceLd + 4 * quad), y[1]);
        y[1] += mfma16(fine[1], lds_quad(M + (16 + c16) * kPieceLd + 16 + 4 * quad), f32x4{0.f, 0.f, 0.f, 0.f});
        const int col = p0 + 16 * wave + 4 * quad;
#pragma unroll
        for (int f = 0; f < 2; ++f) {
          const int t = t0 + 16 * f + c16;
          if (t >= t_last) continue;
          y[f] += carried[f];
          if (a.skip) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (col + r < a.P) y[f][r] = fmaf(skip, VT[token_quad(16 * wave + 4 * quad + r, 4 * f + (c16 >> 2)) + (c16 & 3)], y[f][r]);
          }
          float* o = a.out + (size_t)(q_begin + t) * ((size_t)a.heads * ld) + (size_t)head * ld + col;
          if ((vec & kVecOut) && col + 4 <= ld) {
            *reinterpret_cast<f32x4*>(o) = y[f];
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (col + r < ld) o[r] = y[f][r];
          }
        }
      }
    }
  }
  if (MODE != kChunkOut && p < ld) {
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = 16 * i + 4 * quad + r;
        if (n < a.N) st[(size_t)n * ld + p] = S[i][r];
      }
  }
}

template <int NT, int WAVES, int MODE>
static int launch_pieces(RecurrenceArgs a, const ChunkArgs& ca, int max_chunks, int vec, hipStream_t stream) {
  constexpr size_t lds = (size_t)piece_lds_floats<NT, WAVES, MODE>() * sizeof(float);
  auto kernel = recurrence_piece_kernel<NT, WAVES, MODE>;
  if (lds > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return (int)e;
  }
  a.pblocks = (a.ld + 16 * WAVES - 1) / (16 * WAVES);
  hipLaunchKernelGGL(kernel, dim3(a.heads * a.pblocks, max_chunks), dim3(64 * WAVES), lds, stream, a, ca, vec);
  return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// The same with one decay per head, for heads of up to 256 rows, on the bfloat16 matrix cores: a workgroup walks its chunk in pieces of
// 16 TP tokens.  With D[t, j] the product of the decays of tokens j + 1 .. t of a piece, G_t that of its tokens up to t and S the
// state in front of it,
//   Y = G (Q S) + M V + skip V,   M[t, j] = D[t, j] g_j (q_t . k_j) for j <= t,
//   S <- G_last S + K^T (g_j D[last, j] V).
// A float goes into a product as three bfloat16 numbers that hold all of its 24 bits (float_split.h), a bfloat16 row as itself: QP and VP
// say which q, k and v are.  The products of parts that reach 2^-24 are added in float, the small ones first: one to six
// instructions of 16 x 16 x 32 where the float instruction takes eight of twice the time.
//
// Every product of decays is built by multiplication in 64 bits and rounded once, none from a difference of logarithms.  Inside a tile of 16 tokens D stands in a
// table; from tile to tile it is E_t (from the tile's first token up to t) times the tiles between times F_j (behind j to the end
// of its tile), all factors at most 1.
//
// A wavefront owns 16 columns of S and all of its rows in registers.  A result's lane (g, c) = (lane >> 4, lane & 15) holds rows 4 g ..
// 4 g + 3 of column c: two such tiles of S are the operand of Y^T = S^T Q^T as they stand, when q's rows of 32 lie in the order
// (rows 0-3, 16-19, 4-7, ...).  K lies in LDS by tokens for Q K^T, then, in the same place, by rows for the update.
// All arrays are blocks of four (8 bytes) in an order that spreads the banks.
//
// Values that are no numbers, or round to none in bfloat16, have parts that cancel, and columns of S or of values below 2^-86 lose bits in the third part
// (2^-133 is the smallest bfloat16 number): such columns are walked token by token.  Float rows go in times 2^24 instead, which costs nothing but their
// multiplication.
//
// What bounds it: a piece's chain of barriers, splits and products (the matrix cores a quarter busy) with two wavefronts on a
// SIMD, and beside long chunks the carried states' way through memory.  A prompt of 2,048 tokens, one layer, states + carry + outputs, against
// the same passes with float matrix instructions in pieces of 32 tokens: 64 heads of 128 x 64 in bfloat16 161 -> 76 us (23 + 9 +
// 44), 8 heads of 256 x 512 with float keys 223 -> 160 us (51 + 15 + 94), 8 of 128 x 257 in bfloat16 157 -> 73 us, 16 of 128 x 128 in
// floats 89 -> 81 us; 100 tokens of the first in one workgroup a head 31 -> 21 us.  Errors against 64 bits, 40 to 2,048 tokens at decays from 0.2 to
// 0.999 of six sets of heads: outputs 5.3e-8 to 2.2e-7 (6.4e-8 to 5.0e-7 before, 0.65 of them on average), last states 3.8e-8 to 1.6e-7
// (4.1e-8 to 5.8e-7, 0.52 of them).
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ void note_largest(u16x2& largest, unsigned pair) {          // of two bfloat16 numbers, without their signs
  largest = __builtin_elementwise_max(largest, __builtin_bit_cast(u16x2, pair & 0x7fff7fffu));
}
__device__ __forceinline__ bool no_number(u16x2 largest) { return largest[0] >= 0x7f80 || largest[1] >= 0x7f80; }
// Four floats as three pairs of words of bfloat16 parts, each the rest rounded to nearest.
__device__ __forceinline__ void split4(const f32x4 x, uint2* part, int stride) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    f32x2 rest{x[2 * i], x[2 * i + 1]};
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      const unsigned w = __builtin_bit_cast(unsigned, __builtin_convertvector(rest, bf16x2));
      if (i == 0) part[p * stride].x = w; else part[p * stride].y = w;
      if (p < 2) rest = f32x2{rest[0] - __uint_as_float(w << 16), rest[1] - __uint_as_float(w & 0xffff0000u)};
    }
  }
}
__device__ __forceinline__ bf16x8 octet(uint2 a, uint2 b) { return __builtin_bit_cast(bf16x8, u32x4{a.x, a.y, b.x, b.y}); }

// acc += a b over 32 columns, a in PA parts and b in PB.  SMALL: without the product of the first parts.
template <int PA, int PB, bool SMALL = false>
__device__ __forceinline__ f32x4 multiply_parts(const bf16x8* a, const bf16x8* b, f32x4 acc) {
#pragma unroll
  for (int sum = 2; sum >= (SMALL ? 1 : 0); --sum)                     // the small products first
#pragma unroll
    for (int i = PA - 1; i >= 0; --i) {
      const int j = sum - i;
      if (j >= 0 && j < PB) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc, 0, 0, 0);
    }
  return acc;
}

// Byte offsets of four tokens 4 f .. 4 f + 3 of a row in an array of rows over a piece's T tokens, and of rows n .. n + 3 of a token in an
// array of tokens over NP rows.  Both orders spread a wavefront's reads of sixteen rows and its writes over all banks.
template <int T> __device__ __forceinline__ int by_row_at(int row, int f) {
  if (T == 64) return row * 128 + (((f >> 1) ^ row ^ (row >> 3)) & 7) * 16 + (f & 1) * 8;
  return (row ^ ((row >> 2) & 1)) * 64 + (((f >> 1) ^ (row >> 1) ^ (row >> 3)) & 3) * 16 + (f & 1) * 8;
}
template <int NP> __device__ __forceinline__ int by_token_at(int t, int n) {
  const int piece = (n >> 5) * 4 + ((n >> 2) & 3);
  return t * NP * 2 + ((piece & ~7) | ((piece ^ t) & 7)) * 16 + ((n >> 4) & 1) * 8;
}

template <int TP> struct alignas(16) PieceDecays {
  float D[TP][16][20];                                                 // inside the tiles; a tile's row t, its columns j
  float E[16 * TP], F[16 * TP];                                        // (F times g)
  float G[16 * TP], H[16 * TP];                                        // products up to t of the piece; behind j, times g; with the scales of Y and of the update
  float a[16 * TP], g[16 * TP];
  float tiles[TP];                                                     // of whole tiles
  double all;                                                          // of the whole piece
};

template <int NT, int WAVES, int MODE, int TP, int QP, int VP> struct PieceLds {
  static constexpr int kPart = 16 * NT * 16 * TP * 2;                  // bytes of one part of Q or K
  static constexpr int kV = 16 * WAVES * 16 * TP * 2, kM = 16 * TP * 16 * TP * 2;
  static constexpr int kK = 0, kVt = kK + QP * kPart, kQ = kVt + VP * kV, kMt = kQ + (MODE != kChunkState ? QP * kPart : 0),
                       kDecays = kMt + (MODE != kChunkState ? 3 * kM : 0), kOdd = kDecays + 2 * (int)sizeof(PieceDecays<TP>), kBytes = kOdd + 16;
};

template <int NT, int WAVES, int MODE, int TP, int QP, int VP>
__global__ __launch_bounds__(64 * WAVES, 2) void recurrence_split_kernel(RecurrenceArgs a, ChunkArgs ca, int vec) {
  using Lds = PieceLds<NT, WAVES, MODE, TP, QP, VP>;
  constexpr int NP = 16 * NT, T = 16 * TP, kThreads = 64 * WAVES;
  constexpr int kBlocks = (NP / 4 * (T / 4) + kThreads - 1) / kThreads, kVBlocks = (4 * WAVES * (T / 4) + kThreads - 1) / kThreads;   // of 4 x 4, a thread's
  constexpr bool kOut = MODE != kChunkState;                           // (kWhole: a sequence from the slot's state to the slot's state)
  // Float rows and M go into products times kScale, which keeps all bits of the smallest (float_split.h), bfloat16 rows and S as they are.  The sums of outputs
  // stand times kOfY; the tables of decays make up for the rest.
  constexpr float kOfK = QP == 1 ? 1.f : kScale, kOfV = VP == 1 ? 1.f : kScale, kOfY = kScale * kOfV, kToM = kScale / (kOfK * kOfK);
  constexpr float kTiny = 0x1p-86f;                                    // columns of S and of values below it lose bits in the third part
  extern __shared__ __attribute__((aligned(16))) unsigned char piece_lds[];
  unsigned char *K = piece_lds + Lds::kK, *VT = piece_lds + Lds::kVt, *Q = piece_lds + Lds::kQ, *M = piece_lds + Lds::kMt;
  PieceDecays<TP>* decays = reinterpret_cast<PieceDecays<TP>*>(piece_lds + Lds::kDecays);
  int* odd = reinterpret_cast<int*>(piece_lds + Lds::kOdd);            // a piece with values that are no numbers; of this piece and the next
  const int tid = threadIdx.x, lane = tid & 63, c16 = lane & 15, quad = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int head = blockIdx.x / a.pblocks, pb = blockIdx.x % a.pblocks;
  int seq = blockIdx.y, local = 0;
  if (MODE != kWhole && !find_chunk(a.cu_seqlens, ca.num_seqs, ca.chunk, blockIdx.y, seq, local)) return;
  const int q_begin = a.cu_seqlens[seq], q_len = a.cu_seqlens[seq + 1] - q_begin;
  if (q_len <= 0) return;
  const int t_first = MODE == kWhole ? 0 : local * ca.chunk, t_last = MODE == kWhole ? q_len : min(t_first + ca.chunk, q_len);
  const int kh = head / (a.heads / a.key_heads), ld = a.ld, p0 = pb * 16 * WAVES;
  const int p = p0 + 16 * wave + c16;                                  // this lane's column of S
  float* st = MODE == kWhole ? a.state + (size_t)a.state_slots[seq] * a.slot_stride + (size_t)head * a.N * ld
                             : ca.ws_state + ((size_t)blockIdx.y * a.heads + head) * a.N * ld;
  const bool from_state = MODE == kChunkOut || (MODE == kWhole && a.seq_starts[seq] > 0);
  const bool live = p0 + 16 * wave < ld;                               // (the wavefront has columns)

  // Memory is read and written through buffers that begin at a place all lanes share: offsets of 32 bits, and where there is nothing to
  // read the offset -1, which gives zeros, so that no load stands behind a branch.
  auto buffer = [](const void* base, size_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(reinterpret_cast<const char*>(base)) + bytes, 0, 0x7fffffff, 0x00027000);
  };
  f32x4 S[NT];
  const __amdgpu_buffer_rsrc_t state = buffer(st, 0);
  const int state_at = p < ld ? (4 * quad * ld + p) * 4 : -1;
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      S[i][r] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(state, from_state && 16 * i + 4 * quad + r < a.N && state_at >= 0 ? state_at + (16 * i + r) * ld * 4 : -1, 0, 0));
  const float skip = a.skip ? a.skip[head] : 0.f;
  const bool skip_in_m = ld == a.P;                                    // (a normaliser's column has no skip)
  const float rate = a.raw ? expf(a.a_log[head]) : 0.f, raw_bias = a.raw ? a.raw_bias[head] : 0.f;

  // The decays of a piece, by the last wavefront: lane 16 i + j has token j of tile i.  What it reads is asked for a piece ahead.
  float raw_a = 1.f, raw_g = 0.f;
  auto ask_decays = [&](int t0) {
    const bool in = lane < min(T, t_last - t0);
    const size_t row = (size_t)(q_begin + t0 + (in ? lane : 0));
    if (a.raw) {
      raw_a = in ? load_as_f32(a.raw, a.raw_dtype, row * a.raw_stride + head) : 0.f;
      raw_g = in ? 1.f : 0.f;
    } else {
      raw_a = in ? a.decay[row * a.decay_stride + head] : 1.f;
      raw_g = !in ? 0.f : a.vscale ? a.vscale[row * a.heads + head] : 1.f;
    }
  };
  auto walk_decays = [&](PieceDecays<TP>& o) {
    float at = raw_a, gt = raw_g;
    if (a.raw) {
      const float z = raw_a + raw_bias, step = z > 20.f ? z : log1pf(expf(z));
      at = raw_g == 0.f ? 1.f : expf(-rate * step);
      gt *= step;
    }
    // In 64 bits, each product rounded once: a rounding of a decay that all rows and columns share stays in a state that remembers long.
    double d = 0.;
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      const float now = __shfl(at, (lane & 48) + t);                   // (by all lanes: the one it comes from among them)
      d = c16 == t ? 1. : d * now;
      if (lane < T) o.D[quad][t][c16] = (float)d;
    }
    double e = at;                                                     // the products from the tile's first token on
    auto before = [&](auto shift) {
      const uint2 w = __builtin_bit_cast(uint2, e);
      const uint2 from{(unsigned)__builtin_amdgcn_update_dpp(0, (int)w.x, 0x110 + decltype(shift)::value, 0xf, 0xf, false),
                       (unsigned)__builtin_amdgcn_update_dpp(0x3ff00000, (int)w.y, 0x110 + decltype(shift)::value, 0xf, 0xf, false)};      // (1 where there is none)
      e *= __builtin_bit_cast(double, from);
    };
    before(std::integral_constant<int, 1>{}); before(std::integral_constant<int, 2>{});
    before(std::integral_constant<int, 4>{}); before(std::integral_constant<int, 8>{});
    double up_to = 1., behind = 1., all = 1.;                          // whole tiles in front of and behind this lane's
#pragma unroll
    for (int i = 0; i < TP; ++i) {
      const uint2 of = __builtin_bit_cast(uint2, e);
      const double w = __builtin_bit_cast(double, uint2{(unsigned)__builtin_amdgcn_readlane((int)of.x, 16 * i + 15), (unsigned)__builtin_amdgcn_readlane((int)of.y, 16 * i + 15)});
      if (i < quad) up_to *= w;
      if (i > quad) behind *= w;
      all *= w;
      if (lane == 0) o.tiles[i] = (float)w;
    }
    if (lane == 0) o.all = all;
    if (lane < T) {
      o.E[lane] = (float)e;
      o.F[lane] = (float)(d * gt);
      o.G[lane] = (float)(e * up_to * (kOfY / kOfK));
      o.H[lane] = (float)(d * behind * gt * (1.f / kOfK / kOfV));
      o.a[lane] = at;
      o.g[lane] = gt;
    }
  };

  using Quad = std::conditional_t<QP == 1, uint2, f32x4>;              // four elements of a row as they are fetched
  using VQuad = std::conditional_t<VP == 1, uint2, f32x4>;
  // Elements n .. n + 3 of a row, zeros past its end.
  auto ask = [](auto& to, const __amdgpu_buffer_rsrc_t& from, int dtype, int at, int count, bool wide) {    // `at`: in elements; count: elements there are, from `at` on
    if (dtype == PLLM_F32) {
      f32x4 x;
      if (wide) {
        x = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(from, count > 0 ? 4 * at : -1, 0, 0));
      } else {
#pragma unroll
        for (int u = 0; u < 4; ++u) x[u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(from, count > u ? 4 * (at + u) : -1, 0, 0));
      }
      if constexpr (std::is_same_v<std::remove_reference_t<decltype(to)>, f32x4>) to = x;
    } else {
      uint2 x;
      if (wide) {
        x = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(from, count > 0 ? 2 * at : -1, 0, 0));
      } else {
        unsigned h[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) h[u] = (unsigned)(unsigned short)__builtin_amdgcn_raw_buffer_load_b16(from, count > u ? 2 * (at + u) : -1, 0, 0);
        x = uint2{h[0] | h[1] << 16, h[2] | h[3] << 16};
      }
      if constexpr (std::is_same_v<std::remove_reference_t<decltype(to)>, f32x4>)
        to = f32x4{__uint_as_float(x.x << 16), __uint_as_float(x.x & 0xffff0000u), __uint_as_float(x.y << 16), __uint_as_float(x.y & 0xffff0000u)};
      else to = x;
    }
  };
  Quad rq[kOut ? kBlocks : 1][4], rk[kBlocks][4];
  VQuad rv[kVBlocks][4];
  const int qk_type = QP == 1 ? PLLM_BF16 : a.qk_dtype, v_type = VP == 1 ? PLLM_BF16 : a.v_dtype;
  auto fetch = [&](int t0) {
    const size_t first = (size_t)(q_begin + t0), qk_bytes = qk_type == PLLM_F32 ? 4 : 2, v_bytes = v_type == PLLM_F32 ? 4 : 2;
    const __amdgpu_buffer_rsrc_t ks = buffer(a.k, (first * a.qk_stride + (size_t)kh * a.N) * qk_bytes), qs = buffer(a.q, (first * a.qk_stride + (size_t)kh * a.N) * qk_bytes),
                                 vs = buffer(a.v, (first * a.v_stride + (size_t)head * a.P) * v_bytes);
    const int there = min(T, t_last - t0);
#pragma unroll
    for (int e = 0; e < kBlocks; ++e) {
      const int at = tid + e * kThreads, t = at / (NP / 4) * 4, n = at % (NP / 4) * 4;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int count = t + i < there ? a.N - n : 0, from = (t + i) * a.qk_stride + n;
        ask(rk[e][i], ks, qk_type, from, count, vec & kVecRows);
        if constexpr (kOut) ask(rq[e][i], qs, qk_type, from, count, vec & kVecRows);
      }
    }
#pragma unroll
    for (int e = 0; e < kVBlocks; ++e) {
      const int at = tid + e * kThreads, t = at / (4 * WAVES) * 4, col = p0 + at % (4 * WAVES) * 4;
#pragma unroll
      for (int i = 0; i < 4; ++i) ask(rv[e][i], vs, v_type, (t + i) * a.v_stride + col, t + i < there ? a.P - col : 0, vec & kVecValues);
    }
  };
  // A block's parts by tokens (to[part][token]) and the same transposed (parts of the four tokens of a row).
  auto parts_of = [&](const auto* raw, uint2 (*to)[4]) {
    if constexpr (std::is_same_v<std::remove_const_t<std::remove_reference_t<decltype(raw[0])>>, uint2>) {
#pragma unroll
      for (int i = 0; i < 4; ++i) to[0][i] = raw[i];
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) split4(raw[i] * kScale, &to[0][i], 4);
    }
  };
  auto check = [&](const uint2* x, int t, int* odd) {                   // a block's tokens with elements that are no numbers
    u16x2 largest{0, 0};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      note_largest(largest, x[i].x);
      note_largest(largest, x[i].y);
    }
    if (no_number(largest)) {
#pragma unroll
      for (int i = 3; i >= 0; --i) {
        u16x2 one{0, 0};
        note_largest(one, x[i].x);
        note_largest(one, x[i].y);
        if (no_number(one)) atomicMin(odd, t + i);
      }
    }
  };
  auto transposed = [&](const uint2* x, int i) {                       // row i of a block of four tokens
    const unsigned pick = i & 1 ? 0x07060302u : 0x05040100u;
    return i < 2 ? uint2{__builtin_amdgcn_perm(x[1].x, x[0].x, pick), __builtin_amdgcn_perm(x[3].x, x[2].x, pick)}
                 : uint2{__builtin_amdgcn_perm(x[1].y, x[0].y, pick), __builtin_amdgcn_perm(x[3].y, x[2].y, pick)};
  };
  auto put = [](unsigned char* at, uint2 v) { *reinterpret_cast<uint2*>(at) = v; };
  auto get = [](const unsigned char* at) { return *reinterpret_cast<const uint2*>(at); };
  auto get8 = [](const unsigned char* at) { return *reinterpret_cast<const bf16x8*>(at); };

  if (kOut)
    for (int i = tid; i < 3 * Lds::kM / 16; i += kThreads) reinterpret_cast<u32x4*>(M)[i] = u32x4{0u, 0u, 0u, 0u};   // (late keys' tiles stay zero)
  if (tid < 2) odd[tid] = T;
  if (wave == WAVES - 1) ask_decays(t_first);
  fetch(t_first);
  if (wave == WAVES - 1) walk_decays(decays[0]);
  double total = 1.;                                                   // first pass: the product of the chunk's decays

  for (int t0 = t_first, turn = 0; t0 < t_last; t0 += T, turn ^= 1) {
    const bool last = t0 + T >= t_last;
    const PieceDecays<TP>& dec = decays[turn];
    uint2 kt[kBlocks][QP][4];
    __syncthreads();                                                   // the piece before is done with LDS
#pragma unroll
    for (int e = 0; e < kBlocks; ++e) {
      const int at = tid + e * kThreads, t = at / (NP / 4) * 4, n = at % (NP / 4) * 4;
      parts_of(rk[e], kt[e]);
      check(kt[e][0], t, odd + turn);
      if (NP * T / 16 % kThreads && t >= T) break;
      if constexpr (kOut) {
        uint2 qt[QP][4];
        parts_of(rq[e], qt);
        check(qt[0], t, odd + turn);
#pragma unroll
        for (int part = 0; part < QP; ++part)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            put(K + part * Lds::kPart + by_token_at<NP>(t + i, n), kt[e][part][i]);
            put(Q + part * Lds::kPart + by_token_at<NP>(t + i, n), qt[part][i]);
          }
      } else {
#pragma unroll
        for (int part = 0; part < QP; ++part)
#pragma unroll
          for (int i = 0; i < 4; ++i) put(K + part * Lds::kPart + by_row_at<T>(n + i, t >> 2), transposed(kt[e][part], i));
      }
    }
#pragma unroll
    for (int e = 0; e < kVBlocks; ++e) {
      const int at = tid + e * kThreads, t = at / (4 * WAVES) * 4, col = at % (4 * WAVES) * 4;
      uint2 vt[VP][4];
      parts_of(rv[e], vt);
      if (ld > a.P && ((p0 + col) ^ a.P) < 4) {                        // the normaliser's column
        const unsigned one = (VP == 1 ? 0x3f80u : 0x4b80u) << ((a.P & 1) * 16);       // (1 or 2^24)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (t0 + t + i < t_last) {
            if (a.P & 2) vt[0][i].y |= one; else vt[0][i].x |= one;
          }
      }
      if (WAVES * T % kThreads && t >= T) break;
#pragma unroll
      for (int part = 0; part < VP; ++part)
#pragma unroll
        for (int i = 0; i < 4; ++i) put(VT + part * Lds::kV + by_row_at<T>(col + i, t >> 2), transposed(vt[part], i));
    }
    __syncthreads();
    constexpr bool kAskLate = kOut && NT > 8;                           // (beside what the transposed keys take there are no registers)
    if (!kAskLate && !last) fetch(t0 + T);
    if (wave == WAVES - 1 && !last) ask_decays(t0 + T);

    f32x4 y[TP];
    bool odd_state = false;                                            // this lane's rows of S
    if constexpr (kOut) {
      for (int id = wave; id < TP * (TP + 1) / 2; id += WAVES) {       // tiles of M on and below the diagonal
        const int tt = id < 1 ? 0 : id < 3 ? 1 : id < 6 ? 2 : 3, jt = id - tt * (tt + 1) / 2;
        f32x4 m[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
        const int j = 16 * jt + 4 * quad, t = 16 * tt + c16;
#pragma unroll
        for (int s = 0; s < NT / 2; ++s) {
          if (NT > 8 && s % 2 == 0) __builtin_amdgcn_sched_barrier(0);             // (reads too far ahead cost registers)
          bf16x8 kf[QP], qf[QP];
#pragma unroll
          for (int part = 0; part < QP; ++part) {
            kf[part] = get8(K + part * Lds::kPart + by_token_at<NP>(16 * jt + c16, 32 * s + 4 * quad));
            qf[part] = get8(Q + part * Lds::kPart + by_token_at<NP>(t, 32 * s + 4 * quad));
          }
          if (QP == 1) {
            m[s & 1] = multiply_parts<QP, QP>(kf, qf, m[s & 1]);
          } else {                                                     // (the small products by themselves: fewer roundings of the large sum)
            m[0] = multiply_parts<1, 1>(kf, qf, m[0]);
            m[1] = multiply_parts<QP, QP, true>(kf, qf, m[1]);
          }
        }
        m[0] += m[1];
        if (jt == tt) {
          const f32x4 d = lds_quad(&dec.D[tt][c16][4 * quad]), g = lds_quad(&dec.g[j]);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            m[0][r] = j + r <= t ? m[0][r] * (d[r] * kToM) * g[r] : 0.f;
            if (skip_in_m && j + r == t) m[0][r] = fmaf(skip, kScale, m[0][r]);
          }
        } else {
          float from = dec.E[t] * kToM;
          for (int i = jt + 1; i < tt; ++i) from *= dec.tiles[i];
          m[0] *= lds_quad(&dec.F[j]) * from;
        }
        uint2 part[3];
        u16x2 largest{0, 0};
        split4(m[0], part, 1);
        note_largest(largest, part[0].x);
        note_largest(largest, part[0].y);
        if (no_number(largest)) atomicMin(odd + turn, t);
#pragma unroll
        for (int i = 0; i < 3; ++i) put(M + i * Lds::kM + by_row_at<T>(t, 4 * jt + quad), part[i]);
      }
      constexpr int kSums = TP == 2 ? 2 : 1;
      f32x4 sums[kSums][TP];
#pragma unroll
      for (int i = 0; i < kSums; ++i)
#pragma unroll
        for (int f = 0; f < TP; ++f) sums[i][f] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (live) {
        u16x2 largest{0, 0};
#pragma unroll
        for (int s = 0; s < NT / 2; ++s) {
          if (NT > 8) __builtin_amdgcn_sched_barrier(0);
          uint2 lo[3], hi[3];
          split4(S[2 * s], lo, 1);
          split4(S[2 * s + 1], hi, 1);
          note_largest(largest, lo[0].x); note_largest(largest, lo[0].y);
          note_largest(largest, hi[0].x); note_largest(largest, hi[0].y);
          const bf16x8 sf[3] = {octet(lo[0], hi[0]), octet(lo[1], hi[1]), octet(lo[2], hi[2])};
#pragma unroll
          for (int f = 0; f < TP; ++f) {
            bf16x8 qf[QP];
#pragma unroll
            for (int part = 0; part < QP; ++part) qf[part] = get8(Q + part * Lds::kPart + by_token_at<NP>(16 * f + c16, 32 * s + 4 * quad));
            sums[s % kSums][f] = multiply_parts<3, QP>(sf, qf, sums[s % kSums][f]);
          }
        }
        odd_state = no_number(largest);
        int most = max((int)largest[0], (int)largest[1]);
        if (__ballot(most > 0 && most < (127 - 86) << 7)) {
          most = max(most, __shfl_xor(most, 16));
          most = max(most, __shfl_xor(most, 32));
          odd_state = odd_state || (most > 0 && most < (127 - 86) << 7);
        }
      }
#pragma unroll
      for (int f = 0; f < TP; ++f) y[f] = (kSums == 2 ? sums[0][f] + sums[kSums - 1][f] : sums[0][f]) * dec.G[16 * f + c16];
      __syncthreads();                                                 // M is whole; K has been read by tokens
#pragma unroll
      for (int e = 0; e < kBlocks; ++e) {
        const int at = tid + e * kThreads, t = at / (NP / 4) * 4, n = at % (NP / 4) * 4;
        if (NP * T / 16 % kThreads && t >= T) break;
#pragma unroll
        for (int part = 0; part < QP; ++part)
#pragma unroll
          for (int i = 0; i < 4; ++i) put(K + part * Lds::kPart + by_row_at<T>(n + i, t >> 2), transposed(kt[e][part], i));
      }
      __syncthreads();
      if (kAskLate && !last) fetch(t0 + T);
    }
    // Columns with a value that is no number, and all of them from a token on whose key or query has one, are walked token by token
    // behind the products, and keep what the products gave for the tokens before.  S waits where it came from or goes to, in
    // memory that no other workgroup uses meanwhile.
    int first_odd = odd_state ? 0 : odd[turn];
    if (tid == 0) odd[turn ^ 1] = T;                                   // (this piece's word is written again two pieces on)
    {
      u16x2 largest{0, 0};
      u32x4 w[TP / 2];
#pragma unroll
      for (int f = 0; f < TP / 2; ++f) {
        w[f] = *reinterpret_cast<const u32x4*>(VT + by_row_at<T>(16 * wave + c16, 8 * f + 2 * quad));
#pragma unroll
        for (int i = 0; i < 4; ++i) note_largest(largest, w[f][i]);
      }
      if (no_number(largest)) {
#pragma unroll
        for (int f = 0; f < TP / 2; ++f)
#pragma unroll
          for (int i = 0; i < 8; ++i)
            if (((w[f][i >> 1] >> (16 * (i & 1))) & 0x7f80u) == 0x7f80u) first_odd = min(first_odd, 32 * f + 8 * quad + i);
      }
    }
    bool any_odd = __ballot(first_odd < T) != 0;
    auto keep_state = [&](auto to_memory) {
      int first_at = state_at, row = 4 * quad;
      asm volatile("" : "+v"(first_at), "+v"(row));                    // (its offsets are not worth registers outside)
#pragma unroll
      for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int at = 16 * i + row + r < a.N && first_at >= 0 ? first_at + (16 * i + r) * ld * 4 : -1;
          if constexpr (decltype(to_memory)::value) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(S[i][r]), state, at, 0, 0);
          else S[i][r] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(state, at, 0, 0));
        }
    };
    auto whole_column = [&] {                                          // (a column is four lanes')
      first_odd = min(first_odd, __shfl_xor(first_odd, 16));
      first_odd = min(first_odd, __shfl_xor(first_odd, 32));
    };
    if (any_odd) {
      whole_column();
      keep_state(std::true_type{});
    }
    if (kOut && live) {
#pragma unroll
      for (int s = 0; s < TP / 2; ++s) {
        bf16x8 vf[VP];
#pragma unroll
        for (int part = 0; part < VP; ++part) {
          vf[part] = get8(VT + part * Lds::kV + by_row_at<T>(16 * wave + c16, 8 * s + 2 * quad));
          if (any_odd) {                                               // (a weight of zero must not meet a later value that is no number)
            u32x4 w = __builtin_bit_cast(u32x4, vf[part]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              if ((w[i] & 0x7f80u) == 0x7f80u) w[i] &= 0xffff0000u;
              if ((w[i] & 0x7f800000u) == 0x7f800000u) w[i] &= 0xffffu;
            }
            vf[part] = __builtin_bit_cast(bf16x8, w);
          }
        }
#pragma unroll
        for (int f = 2 * s; f < TP; ++f) {
          bf16x8 mf[3];
#pragma unroll
          for (int part = 0; part < 3; ++part) mf[part] = get8(M + part * Lds::kM + by_row_at<T>(16 * f + c16, 8 * s + 2 * quad));
          y[f] = multiply_parts<VP, 3>(vf, mf, y[f]);
        }
      }
      // Outputs past 2^79 leave the scaled floats: from the first of them on as well.
      float none = 0.f;
#pragma unroll
      for (int f = 0; f < TP; ++f)
#pragma unroll
        for (int r = 0; r < 4; ++r) none = fmaf(y[f][r], 0.f, none);
      if (!__all(none == 0.f)) {
        int from = T;
#pragma unroll
        for (int f = 0; f < TP; ++f)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int before = any_odd ? __shfl(first_odd, 4 * quad + r) : T;
            if (!(fabsf(y[f][r]) < INFINITY) && 16 * f + c16 < before) from = min(from, 16 * f + c16);
          }
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) from = min(from, __shfl_xor(from, d));
        if (!any_odd && from < T) keep_state(std::true_type{});
        first_odd = min(first_odd, from);
        any_odd = any_odd || from < T;
      }
    }
    if (live && (MODE != kChunkOut || !last)) {
      bf16x8 vs[TP / 2][3];
      float most = 0.f;
#pragma unroll
      for (int f = 0; f < TP / 2; ++f) {
        f32x4 lo{0.f, 0.f, 0.f, 0.f}, hi = lo;
#pragma unroll
        for (int part = VP - 1; part >= 0; --part) {
          const unsigned char* at = VT + part * Lds::kV + by_row_at<T>(16 * wave + c16, 8 * f + 2 * quad);
          const u32x4 w = *reinterpret_cast<const u32x4*>(at);
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            lo[2 * i] += __uint_as_float(w[i] << 16); lo[2 * i + 1] += __uint_as_float(w[i] & 0xffff0000u);
            hi[2 * i] += __uint_as_float(w[2 + i] << 16); hi[2 * i + 1] += __uint_as_float(w[2 + i] & 0xffff0000u);
          }
        }
        uint2 lp[3], hp[3];
        lo *= lds_quad(&dec.H[32 * f + 8 * quad]);
        hi *= lds_quad(&dec.H[32 * f + 8 * quad + 4]);
#pragma unroll
        for (int i = 0; i < 4; ++i) most = fmaxf(fmaxf(most, fabsf(lo[i])), fabsf(hi[i]));
        split4(lo, lp, 1);
        split4(hi, hp, 1);
#pragma unroll
        for (int part = 0; part < 3; ++part) vs[f][part] = octet(lp[part], hp[part]);
      }
      // Columns of values so small that their last parts are none, or with one that rounds to no bfloat16 number: the state token by token as well (the
      // outputs above do not take these values).
      constexpr float kNone = 0x1.fep127f;
      if (__ballot((most > 0.f && most < kTiny) || most > kNone)) {
        most = fmaxf(most, __shfl_xor(most, 16));
        most = fmaxf(most, __shfl_xor(most, 32));
        const bool odd_values = (most > 0.f && most < kTiny) || most > kNone;
        if (odd_values) first_odd = min(first_odd, T - 1);
        if (__ballot(odd_values)) {
          whole_column();
          if (!any_odd) keep_state(std::true_type{});
          any_odd = true;
        }
      }
      const float all = (float)dec.all;
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        if (NT > 8 && i % 2 == 0) __builtin_amdgcn_sched_barrier(0);
        S[i] *= all;
#pragma unroll
        for (int f = 0; f < TP / 2; ++f) {
          bf16x8 kf[QP];
#pragma unroll
          for (int part = 0; part < QP; ++part) kf[part] = get8(K + part * Lds::kPart + by_row_at<T>(16 * i + c16, 8 * f + 2 * quad));
          S[i] = multiply_parts<QP, 3>(kf, vs[f], S[i]);
        }
      }
    }
    if (kOut && live) {
      const int col = p0 + 16 * wave + 4 * quad;
      const __amdgpu_buffer_rsrc_t out = buffer(a.out, ((size_t)(q_begin + t0) * a.heads + head) * ld * 4);
#pragma unroll
      for (int f = 0; f < TP; ++f) {
        const int t = 16 * f + c16, at = t < t_last - t0 ? (t * a.heads * ld + col) * 4 : -1;
        y[f] *= 1.f / kOfY;
        if (a.skip && !skip_in_m && at >= 0) {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (col + r < a.P) y[f][r] = fmaf(skip, load_as_f32(a.v, a.v_dtype, (size_t)(q_begin + t0 + t) * a.v_stride + (size_t)head * a.P + col + r), y[f][r]);
        }
        if (vec & kVecOut && !any_odd) {
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, y[f]), out, col < ld ? at : -1, 0, 0);
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int before = any_odd ? __shfl(first_odd, 4 * quad + r) : T;
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y[f][r]), out, col + r < ld && at >= 0 && t < before ? at + 4 * r : -1, 0, 0);
          }
        }
      }
    }
    if (any_odd && first_odd < T && p < ld) {                          // (the lanes of one column together)
#pragma unroll 1
      for (int t = 0; t < min(T, t_last - t0); ++t) {                  // (rows as they stand in memory)
        const size_t row = (size_t)(q_begin + t0 + t), qk_at = row * a.qk_stride + (size_t)kh * a.N;
        const float x = p < a.P ? load_as_f32(a.v, a.v_dtype, row * a.v_stride + (size_t)head * a.P + p) : 1.f, xg = x * dec.g[t], at = dec.a[t];
        float dot = 0.f;
#pragma unroll 1
        for (int n = 4 * quad; n < a.N; n += (n & 3) == 3 ? 13 : 1) {
          float* s = st + (size_t)n * ld + p;
          const float next = fmaf(load_as_f32(a.k, a.qk_dtype, qk_at + n), xg, at * *s);
          *s = next;
          if constexpr (kOut) dot = fmaf(next, load_as_f32(a.q, a.qk_dtype, qk_at + n), dot);
        }
        if constexpr (kOut) {
          dot += __shfl_xor(dot, 16);
          dot += __shfl_xor(dot, 32);
          if (quad == 0 && t >= first_odd) a.out[(size_t)(q_begin + t0 + t) * ((size_t)a.heads * ld) + (size_t)head * ld + p] = p < a.P && a.skip ? fmaf(skip, x, dot) : dot;
        }
      }
      keep_state(std::false_type{});
    }
    if (wave == WAVES - 1 && !last) walk_decays(decays[turn ^ 1]);
    if (!kOut && pb == 0 && tid == 0) {
      total *= dec.all;
      if (last) ca.ws_decay[(size_t)blockIdx.y * a.heads + head] = (float)total;
    }
  }
  if (MODE != kChunkOut) {
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(S[i][r]), state, 16 * i + 4 * quad + r < a.N && state_at >= 0 ? state_at + (16 * i + r) * ld * 4 : -1, 0, 0);
  }
}

template <int NT, int WAVES, int MODE, int TP, int QP, int VP>
static int launch_split(RecurrenceArgs a, const ChunkArgs& ca, int max_chunks, int vec, hipStream_t stream) {
  constexpr int lds = PieceLds<NT, WAVES, MODE, TP, QP, VP>::kBytes;
  static_assert(lds <= (WAVES == 8 ? 160 : 80) * 1024, "LDS of a compute unit, or half of it");
  auto kernel = recurrence_split_kernel<NT, WAVES, MODE, TP, QP, VP>;
  if (lds > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return (int)e;
  }
  a.pblocks = (a.ld + 16 * WAVES - 1) / (16 * WAVES);
  hipLaunchKernelGGL(kernel, dim3(a.heads * a.pblocks, max_chunks), dim3(64 * WAVES), lds, stream, a, ca, vec);
  return (int)hipGetLastError();
}

// Pieces of 64 tokens where q and k are bfloat16, of 32 where they come as three parts and LDS holds no more.
template <int NT, int WAVES, int MODE>
static int launch_split_types(const RecurrenceArgs& a, const ChunkArgs& ca, int max_chunks, int vec, hipStream_t stream) {
  const bool v16 = a.v_dtype != PLLM_F32, q16 = a.qk_dtype != PLLM_F32;
  if (q16 && v16) return launch_split<NT, WAVES, MODE, NT <= 8 ? 4 : 2, 1, 1>(a, ca, max_chunks, vec, stream);
  if (v16) return launch_split<NT, WAVES, MODE, 2, 3, 1>(a, ca, max_chunks, vec, stream);
  return launch_split<NT, WAVES, MODE, 2, 3, 3>(a, ca, max_chunks, vec, stream);
}

// Wavefronts (tiles of 16 columns) of a workgroup: eight for tall states and for a decay per row, whose work per piece that
// all columns share is large and whose LDS leaves room for one workgroup; else four, two workgroups to a compute unit (257
// columns, a normaliser's: 55 us as four and one tile over, 75 us in workgroups of five, which do not pair up; 777 tokens).  Small
// states with a decay per row fill their tiles: 100 heads of 32 x 32, 2,048 tokens, 190 us in workgroups of two wavefronts and 286 us
// padded to 64 x 64 (248 us token by token in chunks).
template <int MODE>
static int launch_piece_pass(const RecurrenceArgs& a, const ChunkArgs& ca, int max_chunks, int vec, hipStream_t stream) {
  const int tiles = (a.ld + 15) / 16;
  if (a.row_decay) {
    if (a.N <= 32 && tiles <= 2) return launch_pieces<2, 2, MODE>(a, ca, max_chunks, vec, stream);
    if (a.N <= 64) return tiles <= 4 ? launch_pieces<4, 4, MODE>(a, ca, max_chunks, vec, stream) : launch_pieces<4, 8, MODE>(a, ca, max_chunks, vec, stream);
    return tiles <= 4 ? launch_pieces<8, 4, MODE>(a, ca, max_chunks, vec, stream) : launch_pieces<8, 8, MODE>(a, ca, max_chunks, vec, stream);
  }
  if (a.N > 128) return launch_split_types<16, 8, MODE>(a, ca, max_chunks, vec, stream);
  return a.N > 64 ? launch_split_types<8, 4, MODE>(a, ca, max_chunks, vec, stream) : launch_split_types<4, 4, MODE>(a, ca, max_chunks, vec, stream);
}

// v_cols: P, or P - 1 for a recurrence with a normaliser (v holds P - 1 columns per head; column P - 1 of S holds
// n_t = a_t n_(t-1) + g_t k_t, and the last element of a head's output n_t . q_t).
// chunk == 0: every sequence token by token in one workgroup per (head, block of channels).  chunk < 0: the same in pieces of
// 32 tokens, for states of up to 256 rows (128 with a decay per row).  chunk > 0: the three passes
// over chunks of that many tokens; ws_state holds max_chunks * heads * N * P floats and ws_decay max_chunks * heads, with
// max_chunks >= sum over the sequences of ceil(q_len / chunk) (total tokens / chunk + num_seqs is enough).
PLLM_API int pllm_linear_recurrence(const void* q, const void* k, int qk_dtype, int qk_stride, const void* v, int v_dtype,
                                    int v_stride, const float* decay, int decay_stride, const float* row_decay, int row_decay_stride,
                                    const float* vscale, const float* skip,
                                    const void* raw, int raw_dtype, int raw_stride, const float* raw_bias, const float* a_log,
                                    float* state, long slot_stride, const int* state_slots, const int* seq_starts,
                                    const int* cu_seqlens, float* out, int num_seqs, int heads, int key_heads, int N, int P,
                                    int v_cols, int chunk, int max_chunks, float* ws_state, float* ws_decay, hipStream_t stream) {
  if (num_seqs <= 0) return 0;
  if (heads <= 0 || key_heads <= 0 || heads % key_heads || N <= 0 || N > 1024 || P <= 0 || (v_cols != P && v_cols != P - 1)) return -2;
  if ((raw && (!raw_bias || !a_log)) || (!raw && !decay && !row_decay) || (row_decay && (raw || decay || heads != key_heads))) return -2;
  if ((chunk > 0 && (max_chunks <= 0 || max_chunks > 65535 || !ws_state || !ws_decay)) || num_seqs > 65535) return -2;
  RecurrenceArgs a;
  a.q = q; a.k = k; a.v = v; a.decay = decay; a.row_decay = row_decay; a.row_decay_stride = row_decay_stride; a.vscale = vscale; a.skip = skip; a.state = state;
  a.state_slots = state_slots; a.seq_starts = seq_starts; a.cu_seqlens = cu_seqlens; a.out = out;
  a.slot_stride = slot_stride; a.qk_dtype = qk_dtype; a.qk_stride = qk_stride; a.v_dtype = v_dtype; a.v_stride = v_stride;
  a.raw = raw; a.raw_dtype = raw_dtype; a.raw_stride = raw_stride; a.raw_bias = raw_bias; a.a_log = a_log;
  a.decay_stride = decay_stride; a.heads = heads; a.key_heads = key_heads; a.N = N; a.P = v_cols; a.ld = P; a.pblocks = (v_cols + 63) / 64;
  ChunkArgs ca{ws_state, ws_decay, chunk, num_seqs};
  const int waves = (N + 63) / 64, need = (N + waves - 1) / waves;   // rows of S per wave
  // (the pieces' kernels count with 32 bits inside a piece)
  const bool near = qk_stride < (1 << 22) && v_stride < (1 << 22) && (long)heads * P < (1 << 22) && (long)N * P < (1l << 29), pieces = near && N <= (row_decay ? 128 : 256);
  auto wide = [](const void* p, int dtype, long stride) { return (reinterpret_cast<uintptr_t>(p) & (dtype == PLLM_F32 ? 15 : 7)) == 0 && stride % 4 == 0; };
  const int vec = (N % 4 == 0 && wide(q, qk_dtype, qk_stride) && wide(k, qk_dtype, qk_stride) ? kVecRows : 0) |
                  (v_cols % 4 == 0 && wide(v, v_dtype, v_stride) ? kVecValues : 0) | (P % 4 == 0 && wide(out, PLLM_F32, 0) ? kVecOut : 0) |
                  (row_decay && N % 4 == 0 && wide(row_decay, PLLM_F32, row_decay_stride) ? kVecDecay : 0);
  if (chunk < 0 && (pieces || near)) {
    if (!pieces) return -2;
    return launch_piece_pass<kWhole>(a, ca, num_seqs, vec, stream);
  }
  if (chunk <= 0) {
    launch_recurrence<kWhole>(a, ca, dim3(heads * a.pblocks, num_seqs), waves, need, stream);
  } else {
    if (pieces) {
      const int code = launch_piece_pass<kChunkState>(a, ca, max_chunks, vec, stream);
      if (code) return code;
    } else {
      launch_recurrence<kChunkState>(a, ca, dim3(heads * a.pblocks, max_chunks), waves, need, stream);
    }
    const size_t per_seq = (size_t)heads * N * P;     // (P: all columns of a row of S, the normaliser's among them)
    hipLaunchKernelGGL(recurrence_carry_kernel, dim3((unsigned)((per_seq + 255) / 256), num_seqs), dim3(256), 0, stream, a, ca);
    if (pieces) {
      const int code = launch_piece_pass<kChunkOut>(a, ca, max_chunks, vec, stream);
      if (code) return code;
    } else {
      launch_recurrence<kChunkOut>(a, ca, dim3(heads * a.pblocks, max_chunks), waves, need, stream);
    }
  }
  PLLM_RETURN_LAST_ERROR();
}

// ---------------------------------------------------------------------------------------------
// decay[t, h] = exp(-exp(A_log[h]) * dt),  dt[t, h] = softplus(raw[t, h] + bias[h])  (no clamp), both float.
template <typename T>
__global__ void step_sizes_kernel(const T* __restrict__ raw, int raw_stride, const float* __restrict__ bias,
                                  const float* __restrict__ a_log, float* __restrict__ dt, float* __restrict__ decay,
                                  int num_tokens, int heads) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= num_tokens * heads) return;
  const int t = idx / heads, h = idx % heads;
  const float z = to_f32(raw[(size_t)t * raw_stride + h]) + bias[h];
  const float step = z > 20.f ? z : log1pf(expf(z));
  dt[idx] = step;
  decay[idx] = expf(-expf(a_log[h]) * step);
}

PLLM_API int pllm_step_sizes(int dtype, const void* raw, int raw_stride, const float* bias, const float* a_log, float* dt,
                             float* decay, int num_tokens, int heads, hipStream_t stream) {
  if (num_tokens <= 0 || heads <= 0) return 0;
  dim3 block(256), grid((num_tokens * heads + 255) / 256);
  if (dtype == PLLM_F32)
    hipLaunchKernelGGL(step_sizes_kernel<float>, grid, block, 0, stream, (const float*)raw, raw_stride, bias, a_log, dt, decay, num_tokens, heads);
  else
    hipLaunchKernelGGL(step_sizes_kernel<bf16>, grid, block, 0, stream, (const bf16*)raw, raw_stride, bias, a_log, dt, decay, num_tokens, heads);
  PLLM_RETURN_LAST_ERROR();
}

// ---------------------------------------------------------------------------------------------
// Behind a recurrence: y [T, inner] float, gate [T, inner] (row stride gate_stride), groups of `group` channels.
//   gate_first:   u = y * silu(gate);  out = u / sqrt(mean_group(u^2) + eps) * w
//   otherwise:    out = y / sqrt(mean_group(y^2) + eps) * silu(gate) [* w]
// One workgroup per token.  With at least as many groups as waves each wave takes whole groups; else the workgroup
// takes the groups one after the other.
template <typename T>
__global__ __launch_bounds__(256) void gated_group_norm_kernel(const float* __restrict__ y, const T* __restrict__ gate,
                                                               int gate_stride, const float* __restrict__ w, T* __restrict__ out,
                                                               int inner, int group, int gate_first, int gate_act, float eps) {
  __shared__ float scratch[16];
  const int row = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const int groups = inner / group;
  const float* yr = y + (size_t)row * inner;
  const T* gr = gate + (size_t)row * gate_stride;
  T* orow = out + (size_t)row * inner;
  const bool by_wave = groups >= waves;
  const int first = by_wave ? wave : 0, step = by_wave ? waves : 1;
  const int i0 = by_wave ? lane : threadIdx.x, di = by_wave ? 64 : blockDim.x;
  for (int g = first; g < groups; g += step) {
    const int base = g * group;
    float ss = 0.f;
    for (int i = i0; i < group; i += di) {
      float u = yr[base + i];
      if (gate_first && gate_act != kGateNone) u *= gate_f32(to_f32(gr[base + i]), gate_act);
      ss = fmaf(u, u, ss);
    }
    ss = by_wave ? wave_sum(ss) : block_sum(ss, scratch);
    const float inv = 1.f / sqrtf(ss / (float)group + eps);
    for (int i = i0; i < group; i += di) {
      const float s = gate_act == kGateNone ? 1.f : gate_f32(to_f32(gr[base + i]), gate_act);
      float u = yr[base + i];
      u = gate_first ? (u * s) * inv : (u * inv) * s;
      if (w) u *= w[base + i];
      orow[base + i] = from_f32<T>(u);
    }
  }
}

// The same for groups whose channels a wave (or, with fewer groups than waves, a few waves side by side) holds in
// registers: every value is read once, four channels per lane and load.  Needs group % 4 == 0, rows that start on
// 16-byte (float) and 8-byte (bfloat16) boundaries, and at most kGroupRegs * 256 channels per wave.
// All of a group's loads are asked for before the first is used (with the gate's conversion beside each load they waited in turn, and the
// weights' for the sum): QUADS is the fewest of 1, 2, 4 and 8 that hold a wave's channels.  What bounds it: memory (8 bytes a channel with a
// bfloat16 gate: 4.1 to 4.5 TB/s at 2,048 rows).  us in turn and at once: 2,048 rows of 4,096 channels 21.2 and 16.5, in groups of 512 20.7
// and 14.9; 777 of 2,048 in groups of 256 6.1 and 5.7; 301 of 8,192 11.7 and 8.7; 8 of 4,096 6.3 and 4.5.
constexpr int kGroupRegs = 8;

template <typename T, int QUADS>
__global__ __launch_bounds__(256) void gated_group_norm_regs_kernel(const float* __restrict__ y, const T* __restrict__ gate,
                                                                    int gate_stride, const float* __restrict__ w, T* __restrict__ out,
                                                                    int inner, int group, int gate_first, int gate_act, float eps) {
  __shared__ float scratch[4];
  const int row = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int groups = inner / group;
  const int parts = groups >= 4 ? 1 : 4 / groups;          // waves side by side on one group (groups 1 or 2; 3 gives 1)
  const int slice = group / parts;                         // channels of a group that one wave takes
  const float* yr = y + (size_t)row * inner;
  const T* gr = gate + (size_t)row * gate_stride;
  T* orow = out + (size_t)row * inner;
  for (int g = wave / parts; g < groups; g += 4 / parts) {
    const int base = g * group + (wave % parts) * slice;
    Quad<float> yv[QUADS], wv[QUADS];
    Quad<T> gv[QUADS];
#pragma unroll
    for (int j = 0; j < QUADS; ++j) yv[j] = *reinterpret_cast<const Quad<float>*>(yr + base + min((j * 64 + lane) * 4, slice - 4));
    if (gate_act != kGateNone) {
#pragma unroll
      for (int j = 0; j < QUADS; ++j) gv[j] = *reinterpret_cast<const Quad<T>*>(gr + base + min((j * 64 + lane) * 4, slice - 4));
    }
    if (w) {
#pragma unroll
      for (int j = 0; j < QUADS; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) wv[j].v[e] = w[base + min((j * 64 + lane) * 4, slice - 4) + e];
    }
    float u[QUADS][4], s[QUADS][4];
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < QUADS; ++j)
      if ((j * 64 + lane) * 4 < slice) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          s[j][e] = gate_act == kGateNone ? 1.f : gate_f32(to_f32(gv[j].v[e]), gate_act);
          u[j][e] = gate_first ? yv[j].v[e] * s[j][e] : yv[j].v[e];
          ss = fmaf(u[j][e], u[j][e], ss);
        }
      }
    ss = wave_sum(ss);
    if (parts > 1) {                                       // (then every wave runs this loop exactly once)
      scratch[wave] = ss;
      __syncthreads();
      ss = 0.f;
      for (int k = 0; k < parts; ++k) ss += scratch[(wave / parts) * parts + k];
    }
    const float inv = 1.f / sqrtf(ss / (float)group + eps);
#pragma unroll
    for (int j = 0; j < QUADS; ++j) {
      const int at = (j * 64 + lane) * 4;
      if (at < slice) {
        Quad<T> o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float r = gate_first ? u[j][e] * inv : (u[j][e] * inv) * s[j][e];
          if (w) r *= wv[j].v[e];
          o.v[e] = from_f32<T>(r);
        }
        *reinterpret_cast<Quad<T>*>(orow + base + at) = o;
      }
    }
  }
}

// The same for small groups, whose lanes (four channels each, a power of two of them, at most 32) lie side by side in a
// wavefront: every lane works, where the kernel above would leave most of a wavefront without channels.
template <typename T>
__global__ __launch_bounds__(256) void gated_group_norm_lanes_kernel(const float* __restrict__ y, const T* __restrict__ gate,
                                                                     int gate_stride, const float* __restrict__ w, T* __restrict__ out,
                                                                     int inner, int group, int gate_first, int gate_act, float eps) {
  const int row = blockIdx.y, at = 4 * (blockIdx.x * blockDim.x + threadIdx.x), lanes = group / 4;
  const bool in = at < inner;                                // (inner is a multiple of the group: a group is in or out as a whole)
  float u[4] = {0.f, 0.f, 0.f, 0.f}, s[4] = {1.f, 1.f, 1.f, 1.f};
  float ss = 0.f;
  if (in) {
    const float4 yv = *reinterpret_cast<const float4*>(y + (size_t)row * inner + at);
    u[0] = yv.x; u[1] = yv.y; u[2] = yv.z; u[3] = yv.w;
    if (gate_act != kGateNone) {
      const Quad<T> gv = *reinterpret_cast<const Quad<T>*>(gate + (size_t)row * gate_stride + at);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] = gate_f32(to_f32(gv.v[e]), gate_act);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (gate_first) u[e] *= s[e];
      ss = fmaf(u[e], u[e], ss);
    }
  }
  for (int off = 1; off < lanes; off <<= 1) ss += __shfl_xor(ss, off, 64);
  if (!in) return;
  const float inv = 1.f / sqrtf(ss / (float)group + eps);
  Quad<T> o;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float r = gate_first ? u[e] * inv : (u[e] * inv) * s[e];
    if (w) r *= w[at + e];
    o.v[e] = from_f32<T>(r);
  }
  *reinterpret_cast<Quad<T>*>(out + (size_t)row * inner + at) = o;
}

static bool group_norm_in_lanes(int inner, int group, int num_tokens) {
  const int lanes = group / 4;
  return group <= 128 && (lanes & (lanes - 1)) == 0 && inner / group >= 4 && num_tokens <= 65535;
}

template <typename T>
static bool group_norm_in_registers(const float* y, const void* gate, int gate_stride, void* out, int inner, int group) {
  const int groups = inner / group, parts = groups >= 4 ? 1 : 4 / groups;
  return group % (4 * parts) == 0 && group / parts <= kGroupRegs * 256 && inner % 4 == 0 && gate_stride % 4 == 0 &&
         (uintptr_t)y % 16 == 0 && (uintptr_t)gate % (4 * sizeof(T)) == 0 && (uintptr_t)out % (4 * sizeof(T)) == 0;
}

template <typename T>
static void launch_group_norm_regs(const float* y, const void* gate, int gate_stride, const float* w, void* out, int num_tokens, int inner, int group,
                                   int gate_first, int gate_act, float eps, hipStream_t stream) {
  const int groups = inner / group, slice = group / (groups >= 4 ? 1 : 4 / groups);
#define PLLM_NORM(QUADS) hipLaunchKernelGGL((gated_group_norm_regs_kernel<T, QUADS>), dim3(num_tokens), dim3(256), 0, stream, y, (const T*)gate, gate_stride, w, \
                                            (T*)out, inner, group, gate_first, gate_act, eps)
  if (slice <= 256) PLLM_NORM(1); else if (slice <= 512) PLLM_NORM(2); else if (slice <= 1024) PLLM_NORM(4); else PLLM_NORM(kGroupRegs);
#undef PLLM_NORM
}

PLLM_API int pllm_gated_group_norm(int dtype, const float* y, const void* gate, int gate_stride, const float* w, void* out,
                                   int num_tokens, int inner, int group, int gate_first, int gate_act, float eps, hipStream_t stream) {
  if (num_tokens <= 0) return 0;
  if (group <= 0 || inner % group || gate_act < 0 || gate_act > kGateNone || (!gate && gate_act != kGateNone)) return -2;
  dim3 grid(num_tokens), block(256);
  const int quads = (inner + 3) / 4;
  dim3 lanes_block(quads >= 256 ? 256 : (quads + 63) / 64 * 64), lanes_grid((quads + lanes_block.x - 1) / lanes_block.x, num_tokens);
  if (dtype == PLLM_F32) {
    if (group_norm_in_registers<float>(y, gate, gate_stride, out, inner, group) && group_norm_in_lanes(inner, group, num_tokens))
      hipLaunchKernelGGL(gated_group_norm_lanes_kernel<float>, lanes_grid, lanes_block, 0, stream, y, (const float*)gate, gate_stride, w, (float*)out,
                         inner, group, gate_first, gate_act, eps);
    else if (group_norm_in_registers<float>(y, gate, gate_stride, out, inner, group))
      launch_group_norm_regs<float>(y, gate, gate_stride, w, out, num_tokens, inner, group, gate_first, gate_act, eps, stream);
    else
      hipLaunchKernelGGL(gated_group_norm_kernel<float>, grid, block, 0, stream, y, (const float*)gate, gate_stride, w, (float*)out,
                         inner, group, gate_first, gate_act, eps);
  } else {
    if (group_norm_in_registers<bf16>(y, gate, gate_stride, out, inner, group) && group_norm_in_lanes(inner, group, num_tokens))
      hipLaunchKernelGGL(gated_group_norm_lanes_kernel<bf16>, lanes_grid, lanes_block, 0, stream, y, (const bf16*)gate, gate_stride, w, (bf16*)out,
                         inner, group, gate_first, gate_act, eps);
    else if (group_norm_in_registers<bf16>(y, gate, gate_stride, out, inner, group))
      launch_group_norm_regs<bf16>(y, gate, gate_stride, w, out, num_tokens, inner, group, gate_first, gate_act, eps, stream);
    else
      hipLaunchKernelGGL(gated_group_norm_kernel<bf16>, grid, block, 0, stream, y, (const bf16*)gate, gate_stride, w, (bf16*)out,
                         inner, group, gate_first, gate_act, eps);
  }
  PLLM_RETURN_LAST_ERROR();
}

// ---------------------------------------------------------------------------------------------
// Gates of a matrix memory with exponential input gates (mLSTM), per sequence and head, all in float:
//   i_t = cap tanh((raw_i + b_i) / cap),   f_t = log sigmoid(cap tanh((raw_f + b_f) / cap))         (log-domain gates)
//   m_t = max(f_t + m_(t-1), i_t)          a running maximum; m = 0 in front of a sequence's first token
//   decay[t, h] = exp(f_t + m_(t-1) - m_t),   take[t, h] = exp(i_t - m_t),   m_out[t, h] = m_t,
// so that S_t = decay_t S_(t-1) + take_t k_t v_t^T is the memory divided by exp(m_t).  m of a sequence's last token of
// this step stays in state[slot][m_at + h].
// One wavefront per (head, sequence) walks the sequence's tokens in blocks of 64: a lane makes its token's gates, and the
// maxima are a scan over the lanes of the maps m -> max(a + m, b) ((a, b) of later tokens after (a', b') of earlier
// ones is (a' + a, max(b' + a, b))); a lane past the sequence's end holds the identity (0, -inf).
__global__ __launch_bounds__(64) void mlstm_gates_kernel(const void* __restrict__ raw_i, const void* __restrict__ raw_f, int raw_dtype,
                                                         int raw_stride, const float* __restrict__ bias_i, const float* __restrict__ bias_f,
                                                         float cap, float* state, long slot_stride, int m_at,
                                                         const int* __restrict__ state_slots, const int* __restrict__ seq_starts,
                                                         const int* __restrict__ cu_seqlens, float* __restrict__ decay,
                                                         float* __restrict__ take, float* __restrict__ m_out, int heads) {
  const int lane = threadIdx.x, head = blockIdx.x, seq = blockIdx.y;
  const int q_begin = cu_seqlens[seq], q_len = cu_seqlens[seq + 1] - q_begin;
  if (q_len <= 0) return;
  float* st = state + (size_t)state_slots[seq] * slot_stride + m_at + head;
  float m_in = seq_starts[seq] > 0 ? *st : 0.f;
  const float bi = bias_i ? bias_i[head] : 0.f, bf = bias_f ? bias_f[head] : 0.f;
  for (int t0 = 0; t0 < q_len; t0 += 64) {
    const int t = t0 + lane;
    const bool ok = t < q_len;
    const size_t row = (size_t)(q_begin + (ok ? t : q_len - 1));
    float gi = load_as_f32(raw_i, raw_dtype, row * raw_stride + head) + bi;
    float gf = load_as_f32(raw_f, raw_dtype, row * raw_stride + head) + bf;
    if (cap > 0.f) {
      gi = cap * tanhf(gi / cap);
      gf = cap * tanhf(gf / cap);
    }
    gf = fminf(gf, 0.f) - log1pf(expf(-fabsf(gf)));
    float a = ok ? gf : 0.f, b = ok ? gi : -INFINITY;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const float a_p = __shfl_up(a, off, 64), b_p = __shfl_up(b, off, 64);
      if (lane >= off) {
        b = fmaxf(b_p + a, b);
        a = a_p + a;
      }
    }
    const float m_t = fmaxf(a + m_in, b);
    float m_prev = __shfl_up(m_t, 1, 64);
    if (lane == 0) m_prev = m_in;
    if (ok) {
      const size_t at = row * heads + head;
      decay[at] = expf(gf + m_prev - m_t);
      take[at] = expf(gi - m_t);
      m_out[at] = m_t;
    }
    m_in = __shfl(m_t, 63, 64);
  }
  if (lane == 0) *st = m_in;
}

PLLM_API int pllm_mlstm_gates(const void* raw_i, const void* raw_f, int raw_dtype, int raw_stride, const float* bias_i,
                              const float* bias_f, float cap, float* state, long slot_stride, int m_at, const int* state_slots,
                              const int* seq_starts, const int* cu_seqlens, float* decay, float* take, float* m_out, int num_seqs,
                              int heads, hipStream_t stream) {
  if (num_seqs <= 0) return 0;
  if (heads <= 0 || num_seqs > 65535 || !raw_i || !raw_f || !state) return -2;
  hipLaunchKernelGGL(mlstm_gates_kernel, dim3(heads, num_seqs), dim3(64), 0, stream, raw_i, raw_f, raw_dtype, raw_stride, bias_i, bias_f,
                     cap, state, slot_stride, m_at, state_slots, seq_starts, cu_seqlens, decay, take, m_out, heads);
  PLLM_RETURN_LAST_ERROR();
}

// Behind the recurrence of a matrix memory with a normaliser: y [T, heads, P + 1] float holds S_t^T q_t in its first P
// columns and n_t . q_t in the last; m [T, heads] the running maxima.  Per token and head, in float:
//   o = y[:P] qscale / (max(|y[P] qscale|, exp(-m)) + 1e-6);   u = o / sqrt(mean(o^2) + eps) * w[head, :] * sigmoid(gate[head, :]);
// out [T, heads * P] in the type T.  One wavefront per (token, head).
template <typename T>
__global__ __launch_bounds__(64) void mlstm_output_kernel(const float* __restrict__ y, const float* __restrict__ m, const void* __restrict__ gate,
                                                          int gate_dtype, int gate_stride, const float* __restrict__ w, T* __restrict__ out,
                                                          int heads, int P, float qscale, float eps) {
  const int lane = threadIdx.x, tok = blockIdx.x, head = blockIdx.y;
  const float* row = y + ((size_t)tok * heads + head) * (P + 1);
  const float den = fmaxf(fabsf(row[P] * qscale), expf(-m[(size_t)tok * heads + head])) + 1e-6f;
  const float f = qscale / den;
  float sq = 0.f;
  for (int p = lane; p < P; p += 64) {
    const float o = row[p] * f;
    sq = fmaf(o, o, sq);
  }
  const float inv = 1.f / sqrtf(wave_sum(sq) / (float)P + eps);
  for (int p = lane; p < P; p += 64) {
    const size_t c = (size_t)head * P + p;
    const float g = load_as_f32(gate, gate_dtype, (size_t)tok * gate_stride + c);
    out[(size_t)tok * heads * P + c] = from_f32<T>(row[p] * f * inv * (w ? w[c] : 1.f) / (1.f + expf(-g)));
  }
}

PLLM_API int pllm_mlstm_output(int out_dtype, const float* y, const float* m, const void* gate, int gate_dtype, int gate_stride,
                               const float* w, void* out, int num_tokens, int heads, int P, float qscale, float eps, hipStream_t stream) {
  if (num_tokens <= 0) return 0;
  if (heads <= 0 || heads > 65535 || P <= 0) return -2;
  dim3 grid(num_tokens, heads), block(64);
  if (out_dtype == PLLM_F32)
    hipLaunchKernelGGL(mlstm_output_kernel<float>, grid, block, 0, stream, y, m, gate, gate_dtype, gate_stride, w, (float*)out, heads, P, qscale, eps);
  else
    hipLaunchKernelGGL(mlstm_output_kernel<bf16>, grid, block, 0, stream, y, m, gate, gate_dtype, gate_stride, w, (bf16*)out, heads, P, qscale, eps);
  PLLM_RETURN_LAST_ERROR();
}

// ---------------------------------------------------------------------------------------------
// out[t, c] = silu(rows[t, c]) as float for c < cols: the activated q, k and v of a recurrence whose operands stay in float
// from here on.  rows has a row stride of its own and either element type.
__global__ __launch_bounds__(256) void silu_to_float_kernel(const void* __restrict__ rows, int dtype, int stride, float* __restrict__ out,
                                                            int cols, size_t total) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const size_t t = i / cols, c = i - t * cols;
  out[i] = silu_f32(load_as_f32(rows, dtype, t * stride + c));
}

PLLM_API int pllm_silu_to_float(const void* rows, int dtype, int stride, float* out, int num_tokens, int cols, hipStream_t stream) {
  if (num_tokens <= 0 || cols <= 0) return 0;
  const size_t total = (size_t)num_tokens * cols;
  hipLaunchKernelGGL(silu_to_float_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream, rows, dtype, stride, out, cols, total);
  PLLM_RETURN_LAST_ERROR();
}

// A forget gate with a lower bound per channel, whose complement is the key (a recurrence without a key product):
//   f = lower + (1 - lower) * sigmoid(raw_f + bias),   k = 1 - f,   q = silu(raw_q),
// from rows [T, >= 2 channels] laid out [raw_q | raw_f | ...]; out float [3][T][channels] = q, k, f.
__global__ __launch_bounds__(256) void bounded_forget_gates_kernel(const void* __restrict__ rows, int dtype, int stride,
                                                                   const float* __restrict__ bias, const float* __restrict__ lower,
                                                                   float* __restrict__ out, int channels, size_t total) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const size_t t = i / channels, c = i - t * channels;
  const float zq = load_as_f32(rows, dtype, t * stride + c);
  const float zf = load_as_f32(rows, dtype, t * stride + channels + c) + (bias ? bias[c] : 0.f);
  const float lo = lower ? lower[c] : 0.f;
  const float sg = 1.f / (1.f + expf(-zf));
  const float f = lo + (1.f - lo) * sg;
  out[i] = silu_f32(zq);
  out[total + i] = 1.f - f;
  out[2 * total + i] = f;
}

PLLM_API int pllm_bounded_forget_gates(const void* rows, int dtype, int stride, const float* bias, const float* lower, float* out,
                                       int num_tokens, int channels, hipStream_t stream) {
  if (num_tokens <= 0 || channels <= 0) return 0;
  const size_t total = (size_t)num_tokens * channels;
  hipLaunchKernelGGL(bounded_forget_gates_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream, rows, dtype, stride, bias,
                     lower, out, channels, total);
  PLLM_RETURN_LAST_ERROR();
}
