// The Mamba-2 recurrence (state-space duality form).
//
//   S_t = exp(-a dt_t) S_(t-1) + dt_t b_t x_t^T,   y_t = S_t^T c_t + d x_t      (per head, S in float32)
//
// One token (ssm_step_rows_kernel, other state sizes ssm_step_kernel): half a wave, or a wave, per row of the transposed
// state [vdim][state_size], lanes along the state; the convolution, the softplus and their bookkeeping ran in the projection's epilogue.
//
// Many tokens: chunks of 64.  Within a chunk
//   y_i = exp(L_i) S c_i + sum_{j <= i} (c_i . b_j) exp(L_i - L_j) dt_j x_j + d x_i
//   S  <- exp(L_63) S + sum_j exp(L_63 - L_j) dt_j b_j x_j^T
// with L the running sum of -a dt from the chunk's start, all as matrix products:
//  * ssm_conv_kernel: convolution and silu; leaves x and b transposed per chunk (the contraction over
//    tokens reads eight consecutive tokens of one channel) and b, c row-major;
//  * ssm_prepare_kernel: softplus, the running sums (in double, kept as two floats: their differences
//    enter an exponential) and the convolution's last inputs into the ring;
//  * ssm_scores_kernel: c_i . b_j of every chunk and group, shared by the heads of the group;
//  * ssm_state_kernel: the serial part, and nothing else: the state from chunk to chunk, in registers;
//  * ssm_output_kernel: the outputs of all chunks at once, from the states the serial part left.
// Operands that must keep float32 accuracy (the state, decay-weighted inputs and scores) enter the bfloat16
// matrix cores as a high and a low part.
// The position-0 token starts from a zero state and zero history, whatever a slot held before.
#include <algorithm>

#include "dense.h"
#include "dense_common.h"
#include "kernels_internal.h"

namespace llmopt {
namespace {

constexpr int Q = (int)kSsmChunk;
constexpr int kConvTokens = 16;

__device__ __forceinline__ float bf16_at(const uint16_t *p, size_t i) {
  return (float)reinterpret_cast<const __bf16 *>(p)[i];
}

struct SsmWorkspace {
  void *xt;       // T [chunks][inner][Q]
  void *bt;       // T [chunks][groups * np][Q]
  void *b, *c;    // T [chunks * Q][groups * np]
  float *dt;      // [chunks][heads][Q]
  float *sum;     // [chunks][heads][2][Q] (high parts, low parts)
  float *tail;    // [chunks][heads][Q]: dt times the decay to the chunk's end
  float *scores;  // [chunks][groups][Q][Q]
  void *states;   // T [chunks][heads][planes][vdim to 16][np]: every chunk's incoming state, in operand order
  uint32_t chunks, inner, np;
  size_t bytes;
};

size_t aligned(size_t bytes) { return (bytes + 255) & ~(size_t)255; }

SsmWorkspace layout(const SsmArgs &a) {
  SsmWorkspace w = {};
  w.chunks = (a.m + Q - 1) / Q;
  w.inner = a.heads * a.vdim;
  w.np = (a.state_size + 31) / 32 * 32;
  const size_t element = a.f32 ? 4 : 2, tokens = (size_t)w.chunks * Q;
  uint8_t *base = static_cast<uint8_t *>(a.workspace);
  size_t at = 0;
  auto take = [&](size_t bytes) {
    void *p = base ? base + at : nullptr;
    at += aligned(bytes);
    return p;
  };
  w.xt = take(tokens * w.inner * element);
  w.bt = take(tokens * a.groups * w.np * element);
  w.b = take(tokens * a.groups * w.np * element);
  w.c = take(tokens * a.groups * w.np * element);
  w.dt = static_cast<float *>(take(tokens * a.heads * 4));
  w.sum = static_cast<float *>(take(tokens * a.heads * 8));
  w.tail = static_cast<float *>(take(tokens * a.heads * 4));
  w.scores = static_cast<float *>(take((size_t)w.chunks * a.groups * Q * Q * 4));
  w.states = take((size_t)w.chunks * a.heads * ((a.vdim + 15) / 16 * 16) * w.np * 4);  // two bf16 planes or one f32
  w.bytes = at;
  return w;
}

// ---- one token ---------------------------------------------------------------------------------------

constexpr int kStepRows = 4;  // state rows of a wave

__global__ __launch_bounds__(256) void ssm_step_kernel(SsmArgs a) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const uint32_t inner = a.heads * a.vdim, n = a.state_size;
  const uint32_t first = (blockIdx.x * 4 + wave) * kStepRows;
  if (first >= inner) return;
  const bool fresh = a.step[kStatePosition] == 0;
  float *state = a.ssm_state + ((size_t)a.step[kStateSlot] * inner + first) * n;
  const float *x = a.row + inner, *b = x + inner, *c = b + a.groups * n, *dt = c + a.groups * n;
  float y[kStepRows], decay[kStepRows], gain[kStepRows];
  uint32_t group[kStepRows];
#pragma unroll
  for (int r = 0; r < kStepRows; ++r) {
    const uint32_t row = min(first + r, inner - 1), head = row / a.vdim;
    decay[r] = fresh ? 0.0f : expf(-expf(bf16_at(a.a_log, head)) * dt[head]);
    gain[r] = dt[head] * x[row];
    group[r] = head / (a.heads / a.groups);
    y[r] = 0.0f;
  }
  for (uint32_t k = lane; k < n; k += 64) {
    float s[kStepRows];
#pragma unroll
    for (int r = 0; r < kStepRows; ++r) s[r] = fresh || first + r >= inner ? 0.0f : state[(size_t)r * n + k];
#pragma unroll
    for (int r = 0; r < kStepRows; ++r) {
      s[r] = fmaf(decay[r], s[r], gain[r] * b[group[r] * n + k]);
      if (first + r < inner) state[(size_t)r * n + k] = s[r];
      y[r] = fmaf(s[r], c[group[r] * n + k], y[r]);
    }
  }
#pragma unroll
  for (int r = 0; r < kStepRows; ++r) y[r] = wave_sum(y[r]);
#pragma unroll
  for (int r = 0; r < kStepRows; ++r)
    if (lane == r && first + r < inner) {
      const uint32_t row = first + r;
      a.gated[row] = (y[r] + bf16_at(a.d_skip, row / a.vdim) * x[row]) * silu_f32(a.row[row]);
    }
}

// Rows of whole pieces of four values and at most 128 PIECES: 32 lanes a row, a piece or two a lane, so that one trip brings all
// a wave needs.  The kernel above, for all other sizes, waits for two or three trips one after the other (scalars, then the state; the skip and the gate
// behind the sums).  Bound: that trip and the launch.  A token of 32 heads of 64 x 128: 7.9 to 9.3 us -> 3.1 to 3.4.
template <int PIECES>
__global__ __launch_bounds__(256) void ssm_step_rows_kernel(SsmArgs a) {
  const int lane = threadIdx.x & 31;
  const uint32_t inner = a.heads * a.vdim, n = a.state_size, mine = blockIdx.x * 8 + (threadIdx.x >> 5);
  const uint32_t row = min(mine, inner - 1), head = row / a.vdim, group = head / (a.heads / a.groups);
  const float *x = a.row + inner, *b = x + inner, *c = b + a.groups * n, *dt = c + a.groups * n;
  const float value = x[row], step = dt[head], z = a.row[row], log_rate = bf16_at(a.a_log, head), skip = bf16_at(a.d_skip, head);
  f32x4 into[PIECES], from[PIECES], s[PIECES];
#pragma unroll
  for (int p = 0; p < PIECES; ++p) {
    const uint32_t k = min(p * 128u + lane * 4u, n - 4);
    into[p] = *reinterpret_cast<const f32x4 *>(b + group * n + k);
    from[p] = *reinterpret_cast<const f32x4 *>(c + group * n + k);
  }
  const bool fresh = a.step[kStatePosition] == 0;
  float *state = a.ssm_state + ((size_t)a.step[kStateSlot] * inner + row) * n;
#pragma unroll
  for (int p = 0; p < PIECES; ++p) s[p] = *reinterpret_cast<const f32x4 *>(state + min(p * 128u + lane * 4u, n - 4));
  const float decay = fresh ? 0.0f : expf(-expf(log_rate) * step), gain = step * value;
  float y = 0.0f;
#pragma unroll
  for (int p = 0; p < PIECES; ++p) {
    const uint32_t k = p * 128u + lane * 4u;
    if (k >= n) continue;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      s[p][e] = fmaf(decay, fresh ? 0.0f : s[p][e], gain * into[p][e]);
      y = fmaf(s[p][e], from[p][e], y);
    }
    if (mine < inner) *reinterpret_cast<f32x4 *>(state + k) = s[p];
  }
  y += dpp_f32<0xb1>(y);  // the 32 lanes of the row
  y += dpp_f32<0x4e>(y);
  y += dpp_f32<0x141>(y);
  y += dpp_f32<0x140>(y);
  y += __shfl_xor(y, 16, 64);
  if (lane == 0 && mine < inner) a.gated[row] = (y + skip * value) * silu_f32(z);
}

// ---- many tokens ----------------------------------------------------------------------------------------

// TAPS: the convolution's length (0: any length, its inputs read once per tap).
template <typename T, int TAPS>
__global__ __launch_bounds__(256) void ssm_conv_kernel(SsmArgs a, SsmWorkspace w) {
  const uint32_t n = a.state_size, channels = w.inner + 2 * a.groups * n;
  const uint32_t padded = w.inner + 2 * a.groups * w.np;
  const uint32_t p = blockIdx.x * 256 + threadIdx.x;  // channel, the b and c groups padded to np
  if (p >= padded) return;
  const uint32_t t0 = blockIdx.y * kConvTokens;
  // which channel of the convolution this is
  uint32_t channel = p, within = 0, which = 0;  // which: 0 x, 1 b, 2 c
  bool real = true;
  if (p >= w.inner) {
    const uint32_t q = p - w.inner, bc = a.groups * w.np;
    which = 1 + q / bc;
    within = q % bc;
    const uint32_t g = within / w.np, k = within % w.np;
    real = k < n;
    channel = w.inner + (which - 1) * a.groups * n + g * n + k;
  }
  const uint32_t ld = w.inner + channels;
  const T *input = static_cast<const T *>(a.projected) + w.inner + channel;
  const uint32_t position = a.step[kStatePosition];
  const float *ring = a.conv_state + (size_t)a.step[kStateSlot] * a.taps * channels + channel;
  T out[kConvTokens];
  if (real) {
    const float bias = bf16_at(a.conv_bias, channel);
    float sum[kConvTokens];
#pragma unroll
    for (int i = 0; i < kConvTokens; ++i) sum[i] = bias;
    // the input of a token before the step, and of any
    auto before = [&](int t) { return (int64_t)position + t >= 0 ? ring[(size_t)((position + t) % a.taps) * channels] : 0.0f; };
    auto at = [&](int t) { return t < 0 ? before(t) : t < (int)a.m ? to_f32(input[(size_t)t * ld]) : 0.0f; };
    if (TAPS > 0) {
      // All are requested, at tokens of the step, before the first is used: under a test each, one after the other, 2048 tokens
      // of 4352 channels took 24.4 us for 15.3.
      constexpr int BEFORE = TAPS > 0 ? TAPS - 1 : 0;
      static_assert(BEFORE <= kConvTokens, "only the first tokens of a step reach behind it");
      const int last = (int)a.m - 1;
      T raw[kConvTokens + BEFORE];
#pragma unroll
      for (int i = 0; i < kConvTokens + BEFORE; ++i) raw[i] = input[(size_t)(uint32_t)min(max((int)t0 + i - BEFORE, 0), last) * ld];
      float window[kConvTokens + BEFORE];
#pragma unroll
      for (int i = 0; i < kConvTokens + BEFORE; ++i) window[i] = (int)t0 + i - BEFORE <= last ? to_f32(raw[i]) : 0.0f;
      if (t0 == 0) {
#pragma unroll
        for (int i = 0; i < BEFORE; ++i) window[i] = before(i - BEFORE);
      }
#pragma unroll
      for (int tap = 0; tap < TAPS; ++tap) {
        const float weight = bf16_at(a.conv, (size_t)channel * TAPS + tap);
#pragma unroll
        for (int i = 0; i < kConvTokens; ++i) sum[i] = fmaf(weight, window[i + tap], sum[i]);
      }
    } else {
      for (uint32_t tap = 0; tap < a.taps; ++tap) {
        const float weight = bf16_at(a.conv, (size_t)channel * a.taps + tap);
#pragma unroll
        for (int i = 0; i < kConvTokens; ++i) sum[i] = fmaf(weight, at((int)t0 + i - (int)(a.taps - 1 - tap)), sum[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < kConvTokens; ++i) out[i] = t0 + i < a.m ? (T)silu_f32(sum[i]) : (T)0.0f;
  } else {
#pragma unroll
    for (int i = 0; i < kConvTokens; ++i) out[i] = (T)0.0f;
  }
  const uint32_t chunk = t0 / Q, j = t0 % Q;
  if (which != 2) {
    T *target = which == 0 ? static_cast<T *>(w.xt) + ((size_t)chunk * w.inner + p) * Q + j
                           : static_cast<T *>(w.bt) + ((size_t)chunk * a.groups * w.np + within) * Q + j;
    Frag<T> lo, hi;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      lo[i] = out[i];
      hi[i] = out[8 + i];
    }
    reinterpret_cast<Frag<T> *>(target)[0] = lo;
    reinterpret_cast<Frag<T> *>(target)[1] = hi;
  }
  if (which != 0) {
    T *target = static_cast<T *>(which == 1 ? w.b : w.c) + (size_t)t0 * a.groups * w.np + within;
#pragma unroll
    for (int i = 0; i < kConvTokens; ++i) target[(size_t)i * a.groups * w.np] = out[i];
  }
}

// Blocks [0, chunks * ceil(heads / 4)): softplus and running sums, a wave a head and a lane a token.  The
// blocks behind: the step's last `taps` convolution inputs into the ring.
template <typename T>
__global__ __launch_bounds__(256) void ssm_prepare_kernel(SsmArgs a, SsmWorkspace w) {
  const uint32_t head_blocks = (a.heads + 3) / 4;
  if (blockIdx.x < w.chunks * head_blocks) {
    const uint32_t chunk = blockIdx.x / head_blocks, head = blockIdx.x % head_blocks * 4 + (threadIdx.x >> 6);
    if (head >= a.heads) return;
    const int j = threadIdx.x & 63;
    const uint32_t t = chunk * Q + j;
    const float bias = bf16_at(a.dt_bias, head);
    const float step = t < a.m ? softplus_f32(a.dt[(size_t)t * a.heads + head] + bias) : 0.0f;
    double running = -(double)expf(bf16_at(a.a_log, head)) * (double)step;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const double before = __shfl_up(running, d, 64);
      if (j >= d) running += before;
    }
    const double end = __shfl(running, 63, 64);
    const size_t at = (size_t)chunk * a.heads + head;
    const float high = (float)running;
    w.dt[at * Q + j] = step;
    w.tail[at * Q + j] = step * __expf((float)(end - running));
    w.sum[at * 2 * Q + j] = high;
    w.sum[at * 2 * Q + Q + j] = (float)(running - (double)high);
    return;
  }
  const uint32_t channels = w.inner + 2 * a.groups * a.state_size;
  const uint32_t t = a.m - 1 - (blockIdx.x - w.chunks * head_blocks), position = a.step[kStatePosition] + t;
  float *ring = a.conv_state + ((size_t)a.step[kStateSlot] * a.taps + position % a.taps) * channels;
  const T *input = static_cast<const T *>(a.projected) + (size_t)t * (w.inner + channels) + w.inner;
  for (uint32_t c = threadIdx.x; c < channels; c += 256) ring[c] = to_f32(input[c]);
}

template <typename T>
__global__ __launch_bounds__(256) void ssm_scores_kernel(SsmArgs a, SsmWorkspace w) {
  const uint32_t chunk = blockIdx.x, group = blockIdx.y;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, column = lane & 15, quad = lane >> 4;
  const size_t ld = (size_t)a.groups * w.np;
  const T *b = static_cast<const T *>(w.b) + (size_t)chunk * Q * ld + group * w.np + quad * 8;
  const T *c = static_cast<const T *>(w.c) + (size_t)chunk * Q * ld + group * w.np + quad * 8;
  float *scores = w.scores + ((size_t)chunk * a.groups + group) * Q * Q;
  f32x4 acc[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) acc[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  for (uint32_t k = 0; k < w.np; k += 32) {
    const Frag<T> fc = *reinterpret_cast<const Frag<T> *>(c + (size_t)(wave * 16 + column) * ld + k);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      if (t > wave) continue;
      const Frag<T> fb = *reinterpret_cast<const Frag<T> *>(b + (size_t)(t * 16 + column) * ld + k);
      acc[t] = mma(fb, fc, acc[t]);
    }
  }
#pragma unroll
  for (int t = 0; t < 4; ++t)
    *reinterpret_cast<f32x4 *>(scores + (wave * 16 + column) * Q + t * 16 + quad * 4) = acc[t];
}

// A chunk's incoming state as the matrix cores take it: float as it is, bf16 as a high and a low plane, in
// operand order: [16 state rows][32 columns] blocks, lane (column / 8) * 16 + row holding eight columns, so
// that an operand is one contiguous load and the serial part stores whole lines.
template <typename T>
constexpr int kStatePlanes = sizeof(T) == 4 ? 1 : 2;
template <typename T>
__device__ __forceinline__ T *state_block(const SsmArgs &a, const SsmWorkspace &w, uint32_t chunk, uint32_t head,
                                          int plane, uint32_t v0) {
  const size_t rows = (a.vdim + 15) & ~15u;
  return static_cast<T *>(w.states) +
         ((((size_t)chunk * a.heads + head) * kStatePlanes<T> + plane) * rows + v0) * w.np;
}

template <typename T, int NT>
struct StateOperands {
  Frag<T> x[2];      // x^T of the 16 state rows, 32 tokens each
  Frag<T> b[NT][2];  // b^T of the wave's state columns
  f32x8 tail[2];
  float end;
};

// What `uniform` points at, `bytes` further on in this lane: scalar addresses and one offset.
template <typename P>
__device__ __forceinline__ const P *lane_at(const void *uniform, uint32_t bytes) {
  return reinterpret_cast<const P *>(static_cast<const char *>(uniform) + bytes);
}

// The serial part: a workgroup owns 16 state rows of one head, its waves the 16-column tiles wave + 4 t
// (state_size <= 64 NT); the chunks' incoming states go to the workspace.  No exchange between waves.
// Bound by what a wave issues in turn: a chunk's fourteen requests and 250 vector instructions, most for the high and low parts of
// the inputs and of the state.  2048 tokens, 64 heads of 64 rows, 128 columns: 36.4 us; with an address of its own per lane and
// request and an exit behind every chunk, 40.0.  (Without the requests it takes 25.5, without the stores 30.2.)
// A wave of fewer tiles than NT has a loop for as many: under a test per tile the requests would be waited for one by one, and
// the last tile's again in place of one that is not there made float32 inputs' the bound (2048 tokens, 8 heads of 32 rows, 16
// columns 34.8 us for 19.4; 256 columns spilled).
template <typename T, int TILES>
__device__ __forceinline__ void ssm_state_walk(const SsmArgs &a, const SsmWorkspace &w, const int wave) {
  const uint32_t head = blockIdx.x, v0 = blockIdx.y * 16, group = head / (a.heads / a.groups);
  const int lane = threadIdx.x & 63, column = lane & 15, quad = lane >> 4;
  const uint32_t n = a.state_size, slot = a.step[kStateSlot];
  const bool fresh = a.step[kStatePosition] == 0;
  const size_t ld = (size_t)a.groups * w.np;
  // lane: state row v, columns k .. k + 3 of every tile; rows beyond the head's end repeat its last one
  const uint32_t v = v0 + column, v_row = min(v, a.vdim - 1);
  float *saved = a.ssm_state + (((size_t)slot * a.heads + head) * a.vdim + v_row) * n;

  f32x4 state[TILES];
#pragma unroll
  for (int t = 0; t < TILES; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const uint32_t k = (wave + 4 * t) * 16 + quad * 4 + r;
      state[t][r] = !fresh && k < n ? saved[k] : 0.0f;
    }

  const uint32_t x_at = (v_row * Q + quad * 8) * sizeof(T), b_at = (column * Q + quad * 8) * sizeof(T), tail_at = quad * 32;
  auto load = [&](StateOperands<T, TILES> &o, uint32_t chunk) __attribute__((always_inline)) {
    const T *x = static_cast<const T *>(w.xt) + ((size_t)chunk * w.inner + head * a.vdim) * Q;
    const float *tail = w.tail + ((size_t)chunk * a.heads + head) * Q;
    o.end = w.sum[((size_t)chunk * a.heads + head) * 2 * Q + Q - 1];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      o.x[s] = *lane_at<Frag<T>>(x + s * 32, x_at);
      o.tail[s] = *lane_at<f32x8>(tail + s * 32, tail_at);
#pragma unroll
      for (int t = 0; t < TILES; ++t)
        o.b[t][s] = *lane_at<Frag<T>>(
            static_cast<const T *>(w.bt) + ((size_t)chunk * ld + group * w.np + ((uint32_t)wave + 4 * t) * 16) * Q + s * 32, b_at);
    }
  };
  auto step = [&](const StateOperands<T, TILES> &o, uint32_t chunk) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
      typedef T x4 __attribute__((ext_vector_type(4)));
      const uint32_t at = (wave + 4 * t) / 2 * 512 + (((wave + 4 * t) % 2 * 2 + quad / 2) * 16 + column) * 8 + quad % 2 * 4;
      x4 high;
      if constexpr (kStatePlanes<T> == 2) {
        WideFrag<T> pairs;
        pairs.set_pair(0, state[t][0], state[t][1]);
        pairs.set_pair(2, state[t][2], state[t][3]);
        x4 low;
#pragma unroll
        for (int r = 0; r < 4; ++r) high[r] = pairs.hi[r], low[r] = pairs.lo[r];
        *reinterpret_cast<x4 *>(state_block<T>(a, w, chunk, head, 1, v0) + at) = low;
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) high[r] = state[t][r];
      }
      *reinterpret_cast<x4 *>(state_block<T>(a, w, chunk, head, 0, v0) + at) = high;
    }
    const float carry = __expf(o.end);
#pragma unroll
    for (int t = 0; t < TILES; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) state[t][r] *= carry;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      WideFrag<T> fx;
#pragma unroll
      for (int e = 0; e < 8; e += 2) fx.set_pair(e, to_f32(o.x[s][e]) * o.tail[s][e], to_f32(o.x[s][e + 1]) * o.tail[s][e + 1]);
#pragma unroll
      for (int t = 0; t < TILES; ++t) state[t] = mma_wide_b(o.b[t][s], fx, state[t]);
    }
  };

  // operands two chunks ahead (one exit from the loop: with one behind every step the compiler waits for all requests at its head)
  StateOperands<T, TILES> ring[3];
  load(ring[0], 0);
  load(ring[1], min(1u, w.chunks - 1));
  uint32_t chunk = 0;
  for (; chunk + 3 <= w.chunks; chunk += 3) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      load(ring[(i + 2) % 3], min(chunk + i + 2, w.chunks - 1));
      __builtin_amdgcn_sched_barrier(0);  // the requests stay ahead of the arithmetic
      step(ring[i], chunk + i);
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
    if (chunk + i < w.chunks) step(ring[i], chunk + i);
  if (v < a.vdim)
#pragma unroll
    for (int t = 0; t < TILES; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const uint32_t k = (wave + 4 * t) * 16 + quad * 4 + r;
        if (k < n) saved[k] = state[t][r];
      }
}

template <typename T, int NT>
__global__ __launch_bounds__(256, 1) void ssm_state_kernel(SsmArgs a, SsmWorkspace w) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tiles = ((int)w.np / 16 - wave + 3) / 4;  // of this wave (4 NT - 8 < np / 16 <= 4 NT)
  if (tiles >= NT) ssm_state_walk<T, NT>(a, w, wave);
  if constexpr (NT > 1)
    if (tiles == NT - 1) ssm_state_walk<T, NT - 1>(a, w, wave);
  if constexpr (NT > 2)
    if (tiles == NT - 2) ssm_state_walk<T, NT - 2>(a, w, wave);
}

// The parallel part: a workgroup per chunk and head, 16 tokens a wave.  y^T of 16 state rows: the incoming
// state against c, scaled by the decay since the chunk's start, and x^T against the weighted scores of the
// chunk's earlier tokens (the skip connection is one more weight on the token's own input).
template <typename T, int STEPS>
__global__ __launch_bounds__(256) void ssm_output_kernel(SsmArgs a, SsmWorkspace w) {
  const uint32_t chunk = blockIdx.x, head = blockIdx.y, group = head / (a.heads / a.groups);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, column = lane & 15, quad = lane >> 4;
  const size_t ld = (size_t)a.groups * w.np;
  const int token = wave * 16 + column;  // of the lane's output column
  const uint32_t row = chunk * Q + token;
  const size_t at = (size_t)chunk * a.heads + head;
  const float *dt = w.dt + at * Q, *sum = w.sum + at * 2 * Q;
  const float *score = w.scores + (((size_t)chunk * a.groups + group) * Q + token) * Q;
  const T *c = static_cast<const T *>(w.c) + (size_t)row * ld + group * w.np + quad * 8;
  const float skip = bf16_at(a.d_skip, head);
  Frag<T> fc[STEPS];
#pragma unroll
  for (int s = 0; s < STEPS; ++s)
    if (s * 32 < (int)w.np) fc[s] = *reinterpret_cast<const Frag<T> *>(c + s * 32);
  const float own_high = sum[token], own_low = sum[Q + token];
  WideFrag<T> weight[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int j0 = s * 32 + quad * 8;
    const f32x8 sc = *reinterpret_cast<const f32x8 *>(score + j0), d = *reinterpret_cast<const f32x8 *>(dt + j0);
    const f32x8 high = *reinterpret_cast<const f32x8 *>(sum + j0), low = *reinterpret_cast<const f32x8 *>(sum + Q + j0);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float decayed = __expf((own_high - high[e]) + (own_low - low[e])) * d[e];
      const int j = j0 + e;
      weight[s].set(e, j > token ? 0.0f : fmaf(sc[e], decayed, j == token ? skip : 0.0f));
    }
  }
  const float scale = __expf(own_high);
  const uint32_t lane_bytes = lane * 8 * sizeof(T);
  const T *x_head = static_cast<const T *>(w.xt) + ((size_t)chunk * w.inner + head * a.vdim) * Q;
  for (uint32_t v0 = blockIdx.z * 16; v0 < a.vdim; v0 += gridDim.z * 16) {
    // bfloat16: a tile's operands are requested together, at scalar addresses: 31.4 us at the sizes above, where each request waited
    // in front of its product 35.3.  (The next tile's as well: 34.4, fewer waves fit; two workgroups over a head's tiles: 42.3.)
    // float32's take twice the registers, and the waves that no longer fit cost more: 2048 tokens, 48 heads of 64 rows, 256 columns
    // together 74 us, each in front of its product 67; 32 heads of 128 rows, 96 columns 42.1 / 40.4, and 44.2 at scalar addresses.
    constexpr bool TOGETHER = kStatePlanes<T> == 2;
    const auto state_at = [&](int plane, int s) {
      const T *from = state_block<T>(a, w, chunk, head, plane, v0);
      return TOGETHER ? *lane_at<Frag<T>>(from + s * 512, lane_bytes) : reinterpret_cast<const Frag<T> *>(from)[s * 64 + lane];
    };
    const auto x_at = [&](int s) {
      const uint32_t v_row = min(v0 + column, a.vdim - 1);
      if constexpr (TOGETHER) return *lane_at<Frag<T>>(x_head + s * 32, (v_row * Q + quad * 8) * sizeof(T));
      const T *x = static_cast<const T *>(w.xt) + ((size_t)chunk * w.inner + head * a.vdim + v_row) * Q + quad * 8;
      return *reinterpret_cast<const Frag<T> *>(x + s * 32);
    };
    [[maybe_unused]] Frag<T> state[kStatePlanes<T>][STEPS], x[2];
    if constexpr (TOGETHER) {
#pragma unroll
      for (int plane = 0; plane < kStatePlanes<T>; ++plane)
#pragma unroll
        for (int s = 0; s < STEPS; ++s)
          if (s * 32 < (int)w.np) state[plane][s] = state_at(plane, s);
#pragma unroll
      for (int s = 0; s < 2; ++s) x[s] = x_at(s);
      __builtin_amdgcn_sched_barrier(0);  // the requests stay ahead of the arithmetic
    }
    f32x4 high = {0.0f, 0.0f, 0.0f, 0.0f}, low = high, within = high;
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
      if (s * 32 < (int)w.np) {
        high = mma(TOGETHER ? state[0][s] : state_at(0, s), fc[s], high);
        if constexpr (kStatePlanes<T> == 2) low = mma(state[1][s], fc[s], low);
      }
#pragma unroll
    for (int s = 0; s < 2; ++s)
      if (s * 32 <= wave * 16 + 15)  // the others come later than all of the wave's tokens
        within = mma_wide_b(TOGETHER ? x[s] : x_at(s), weight[s], within);
    if (row >= a.m) continue;
    T *out = static_cast<T *>(a.y) + (size_t)row * w.inner + head * a.vdim + v0 + quad * 4;
    typedef T x4 __attribute__((ext_vector_type(4)));
    x4 y;
#pragma unroll
    for (int r = 0; r < 4; ++r) y[r] = (T)fmaf(scale, high[r] + low[r], within[r]);
    if (a.vdim % 4 == 0) {
      if (v0 + quad * 4 < a.vdim) *reinterpret_cast<x4 *>(out) = y;
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (v0 + quad * 4 + r < a.vdim) out[r] = y[r];
    }
  }
}

template <typename T, int NT>
hipError_t run_scan(const SsmArgs &a, const SsmWorkspace &w, hipStream_t stream) {
  ssm_state_kernel<T, NT><<<dim3(a.heads, (a.vdim + 15) / 16), 256, 0, stream>>>(a, w);
  if (hipError_t status = hipGetLastError()) return status;
  const uint32_t blocks = (a.vdim + 15) / 16;
  const uint32_t parts = std::min<uint32_t>(blocks, std::max<uint32_t>(1, 1024 / std::max<uint32_t>(1, w.chunks * a.heads)));
  ssm_output_kernel<T, 2 * NT><<<dim3(w.chunks, a.heads, parts), 256, 0, stream>>>(a, w);
  return hipGetLastError();
}

template <typename T>
hipError_t run_prefill(const SsmArgs &a, hipStream_t stream) {
  const SsmWorkspace w = layout(a);
  const uint32_t padded = w.inner + 2 * a.groups * w.np;
  const dim3 conv_grid((padded + 255) / 256, w.chunks * Q / kConvTokens);
  if (a.taps == 4) ssm_conv_kernel<T, 4><<<conv_grid, 256, 0, stream>>>(a, w);
  else if (a.taps == 3) ssm_conv_kernel<T, 3><<<conv_grid, 256, 0, stream>>>(a, w);
  else ssm_conv_kernel<T, 0><<<conv_grid, 256, 0, stream>>>(a, w);
  if (hipError_t status = hipGetLastError()) return status;
  ssm_prepare_kernel<T><<<w.chunks * ((a.heads + 3) / 4) + std::min(a.m, a.taps), 256, 0, stream>>>(a, w);
  if (hipError_t status = hipGetLastError()) return status;
  ssm_scores_kernel<T><<<dim3(w.chunks, a.groups), 256, 0, stream>>>(a, w);
  if (hipError_t status = hipGetLastError()) return status;
  if (w.np <= 64) return run_scan<T, 1>(a, w, stream);
  if (w.np <= 128) return run_scan<T, 2>(a, w, stream);
  if (w.np <= 256) return run_scan<T, 4>(a, w, stream);
  return hipErrorInvalidValue;
}

}  // namespace

size_t ssm_workspace_bytes(const SsmArgs &a) {
  SsmArgs sized = a;
  sized.workspace = nullptr;
  return layout(sized).bytes;
}

hipError_t launch_ssm_step(const SsmArgs &a, hipStream_t stream) {
  const uint32_t rows = a.heads * a.vdim, per = 4 * kStepRows;
  const bool aligned = ((reinterpret_cast<uintptr_t>(a.row) | reinterpret_cast<uintptr_t>(a.ssm_state)) & 15) == 0;
  if (aligned && a.state_size % 4 == 0 && rows % 4 == 0 && a.state_size <= 256) {  // (b and c lie behind two times `rows` values)
    const auto kernel = a.state_size <= 128 ? ssm_step_rows_kernel<1> : ssm_step_rows_kernel<2>;
    kernel<<<(rows + 7) / 8, 256, 0, stream>>>(a);
    return hipGetLastError();
  }
  ssm_step_kernel<<<(rows + per - 1) / per, 256, 0, stream>>>(a);
  return hipGetLastError();
}

hipError_t launch_ssm_prefill(const SsmArgs &a, hipStream_t stream) {
  return a.f32 ? run_prefill<float>(a, stream) : run_prefill<__bf16>(a, stream);
}

}  // namespace llmopt
