// Small decode-step kernels around the W4A16 linears and the Q8 attention:
// RMSNorm, rotate-half RoPE for Q and K, fp16 embedding gather, broadcasting
// fp16 add, byte copy and the two-step argmax of the LM head.  All of them move
// a few kilobytes per launch at decode sizes and are launch-latency bound; they
// are written for clarity, one wave per row where a row reduction is needed.
#include <algorithm>

#include "kernels.h"
#include "w4_common.h"

namespace llmopt {
namespace {

constexpr int kRowWaves = 4;  // rows (waves) per workgroup of the row kernels

template <typename In>
__device__ __forceinline__ float load_as_float(const In *p, size_t i);
template <>
__device__ __forceinline__ float load_as_float<uint16_t>(const uint16_t *p, size_t i) {
  return half_bits_to_float(p[i]);
}
template <>
__device__ __forceinline__ float load_as_float<float>(const float *p, size_t i) {
  return p[i];
}

// lib/metal_normalization_source.ml:70-91 and lib/metal_w4a16_source.ml:496-526
template <typename In, bool WEIGHT_FIRST>
__global__ __launch_bounds__(kRowWaves * 64) void rms_norm_kernel(const In *input, const uint16_t *weight,
                                                                  uint16_t *output, uint32_t rows,
                                                                  uint32_t width, float epsilon) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t row = blockIdx.x * kRowWaves + (threadIdx.x >> 6);
  if (row >= rows) return;  // whole wave
  const size_t base = (size_t)row * width;
  float square_sum = 0.0f;
  for (uint32_t col = lane; col < width; col += 64) {
    const float value = load_as_float(input, base + col);
    square_sum += value * value;
  }
  square_sum = wave_sum(square_sum);
  const float inverse = rsqrtf(square_sum / (float)width + epsilon);
  for (uint32_t col = lane; col < width; col += 64) {
    const float value = load_as_float(input, base + col);
    const float w = half_bits_to_float(weight[col]);
    output[base + col] = float_to_half_bits(WEIGHT_FIRST ? value * w * inverse : value * inverse * w);
  }
}

// The LM head's normalisation (lib/metal_w4a16_source.ml:1038-1046 keeps
// x * w * inverse in float32 and multiplies it with the dequantised weights).
// The GEMV kernels take fp16 activations, so the float32 value v goes out as
// two fp16 rows, hi = half(v) and lo = half(v - hi): W.hi + W.lo, accumulated
// in float32, differs from W.v by 2^-22 relative instead of the 2^-11 of a
// single fp16 row.  Output rows 2r (hi) and 2r + 1 (lo).
template <typename In>
__global__ __launch_bounds__(kRowWaves * 64) void rms_norm_split_kernel(const In *input, const uint16_t *weight,
                                                                        uint16_t *output, uint32_t rows,
                                                                        uint32_t width, float epsilon) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t row = blockIdx.x * kRowWaves + (threadIdx.x >> 6);
  if (row >= rows) return;  // whole wave
  const size_t base = (size_t)row * width;
  float square_sum = 0.0f;
  for (uint32_t col = lane; col < width; col += 64) {
    const float value = load_as_float(input, base + col);
    square_sum += value * value;
  }
  square_sum = wave_sum(square_sum);
  const float inverse = rsqrtf(square_sum / (float)width + epsilon);
  uint16_t *high = output + (size_t)(2 * row) * width;
  uint16_t *low = high + width;
  for (uint32_t col = lane; col < width; col += 64) {
    const float value = load_as_float(input, base + col) * half_bits_to_float(weight[col]) * inverse;
    const uint16_t high_bits = float_to_half_bits(value);
    high[col] = high_bits;
    low[col] = float_to_half_bits(value - half_bits_to_float(high_bits));
  }
}

// The same for f16 rows of up to 64 * 8 * kRmsVectors values, width a multiple
// of 8: the row and the weights are requested once, 16 bytes per lane, all
// loads in flight together, and stay in registers between the two passes (the
// loop above walks the row one 2-byte load latency at a time, twice).
constexpr int kRmsVectors = 4;

// SPLIT: the two rows of rms_norm_split_kernel.  (The head of one token, K = 2048: 5 us less than by its loops, a load latency
// for every 64 values, twice.)
template <bool WEIGHT_FIRST, bool SPLIT = false>
__global__ __launch_bounds__(kRowWaves * 64) void rms_norm_f16_rows_kernel(const uint16_t *input,
                                                                           const uint16_t *weight,
                                                                           uint16_t *output, uint32_t rows,
                                                                           uint32_t width, float epsilon) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t row = blockIdx.x * kRowWaves + (threadIdx.x >> 6);
  if (row >= rows) return;  // whole wave
  const uint32_t vectors = width / 8;
  const uint4 *in = reinterpret_cast<const uint4 *>(input + (size_t)row * width);
  const uint4 *w = reinterpret_cast<const uint4 *>(weight);
  uint4 x_raw[kRmsVectors], w_raw[kRmsVectors];
#pragma unroll
  for (int v = 0; v < kRmsVectors; ++v) {
    const uint32_t index = lane + 64 * v;
    x_raw[v] = index < vectors ? in[index] : make_uint4(0, 0, 0, 0);
    w_raw[v] = index < vectors ? w[index] : make_uint4(0, 0, 0, 0);
  }
  float square_sum = 0.0f;
#pragma unroll
  for (int v = 0; v < kRmsVectors; ++v) {
    const h8_t x = __builtin_bit_cast(h8_t, x_raw[v]);
#pragma unroll
    for (int e = 0; e < 8; ++e) square_sum += (float)x[e] * (float)x[e];
  }
  square_sum = wave_sum(square_sum);
  const float inverse = rsqrtf(square_sum / (float)width + epsilon);
  uint4 *out = reinterpret_cast<uint4 *>(output + (size_t)row * width * (SPLIT ? 2 : 1));
#pragma unroll
  for (int v = 0; v < kRmsVectors; ++v) {
    const uint32_t index = lane + 64 * v;
    if (index >= vectors) continue;
    const h8_t x = __builtin_bit_cast(h8_t, x_raw[v]);
    const h8_t g = __builtin_bit_cast(h8_t, w_raw[v]);
    h8_t y, low;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float value = (float)x[e], gain = (float)g[e];
      const float result = WEIGHT_FIRST ? value * gain * inverse : value * inverse * gain;
      y[e] = (_Float16)result;
      if (SPLIT) low[e] = (_Float16)(result - (float)y[e]);
    }
    out[index] = __builtin_bit_cast(uint4, y);
    if (SPLIT) out[vectors + index] = __builtin_bit_cast(uint4, low);
  }
}

// lib/metal_normalization_source.ml:765-802
__global__ __launch_bounds__(kRowWaves * 64) void rotary_qk_kernel(RotaryQkArgs a) {
#pragma clang fp contract(off)  // every product and the sum round to half separately
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t row = blockIdx.x * kRowWaves + (threadIdx.x >> 6);
  const uint32_t total_rows = a.batches * (a.q_heads + a.k_heads) * a.tokens;
  if (row >= total_rows) return;
  const uint32_t q_rows = a.batches * a.q_heads * a.tokens;
  const bool is_q = row < q_rows;
  const uint32_t local_row = is_q ? row : row - q_rows;
  const uint32_t heads = is_q ? a.q_heads : a.k_heads;
  const uint32_t batch = local_row / (heads * a.tokens);
  const uint32_t head_token = local_row % (heads * a.tokens);
  const uint32_t head = head_token / a.tokens;
  const uint32_t token = head_token % a.tokens;
  const size_t input_base = ((size_t)(batch * a.tokens + token) * heads + head) * a.width;
  const _Float16 *input = reinterpret_cast<const _Float16 *>(is_q ? a.q_input : a.k_input);
  _Float16 *output = reinterpret_cast<_Float16 *>(is_q ? a.q_output : a.k_output);
  const _Float16 *cosine = reinterpret_cast<const _Float16 *>(a.cosine);
  const _Float16 *sine = reinterpret_cast<const _Float16 *>(a.sine);
  const uint32_t trig_batch = a.trig_batches == 1 ? 0 : batch;
  const size_t trig_base = (size_t)(trig_batch * a.tokens + token) * a.width;
  const size_t output_base = (size_t)local_row * a.width;
  for (uint32_t col = lane; col < a.width; col += 64)
    output[output_base + col] =
        rotate_half_element(input + input_base, cosine + trig_base, sine + trig_base, col, a.half_dimension);
}

// lib/metal_tensor_source.ml:306-320
__global__ void embedding_kernel(EmbeddingArgs a) {
  const size_t gid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t count = (size_t)a.tokens * a.width;
  if (gid >= count) return;
  const uint32_t token = (uint32_t)(gid / a.width);
  const uint32_t dimension = (uint32_t)(gid % a.width);
  const int64_t index = a.indices[token];
  a.output[gid] =
      (index >= 0 && index < (int64_t)a.vocabulary) ? a.weight[(size_t)index * a.width + dimension] : (uint16_t)0;
}

// llmopt_pointwise_offset, lib/metal_tensor_source.ml:1014-1028
__device__ __forceinline__ uint32_t pointwise_offset(uint32_t gid, const PointwiseArgs &a, bool is_left) {
  uint32_t remaining = gid, offset = 0, stride = 1;
  for (int axis = (int)a.rank - 1; axis >= 0; --axis) {
    const uint32_t output_dimension = a.output_shape[axis];
    const uint32_t coordinate = remaining % output_dimension;
    remaining /= output_dimension;
    const uint32_t input_dimension = is_left ? a.left_shape[axis] : a.right_shape[axis];
    offset += (input_dimension == 1 ? 0 : coordinate) * stride;
    stride *= input_dimension;
  }
  return offset;
}

__global__ void add_f16_kernel(PointwiseArgs a) {
  const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= a.count) return;
  const _Float16 left = a.left_scalar
                            ? (_Float16)a.left_f32
                            : reinterpret_cast<const _Float16 *>(a.left)[pointwise_offset(gid, a, true)];
  const _Float16 right = a.right_scalar
                             ? (_Float16)a.right_f32
                             : reinterpret_cast<const _Float16 *>(a.right)[pointwise_offset(gid, a, false)];
  reinterpret_cast<_Float16 *>(a.output)[gid] = left + right;
}

// both operands have the output's shape: 8 halves per thread
__global__ void add_f16_same_shape_kernel(const uint4 *left, const uint4 *right, uint4 *output,
                                          uint32_t vectors) {
  const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= vectors) return;
  const uint4 l = left[gid], r = right[gid];
  uint4 out;
  out.x = as_u32(as_h2(l.x) + as_h2(r.x));
  out.y = as_u32(as_h2(l.y) + as_h2(r.y));
  out.z = as_u32(as_h2(l.z) + as_h2(r.z));
  out.w = as_u32(as_h2(l.w) + as_h2(r.w));
  output[gid] = out;
}

__global__ void copy_vectors_kernel(const u32x4_t *source, u32x4_t *destination, size_t vectors) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < vectors; i += stride)
    destination[i] = __builtin_nontemporal_load(source + i);
}

__global__ void copy_bytes_kernel(const uint8_t *source, uint8_t *destination, size_t bytes) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < bytes; i += stride)
    destination[i] = source[i];
}

struct Candidate {
  float value;
  uint32_t index;
};

__device__ __forceinline__ bool better(float value, uint32_t index, float best_value, uint32_t best_index) {
  return value > best_value || (value == best_value && index < best_index);
}

// 256 (value, index) candidates per row, the record the reference's stage 1
// hands to its reduce kernel (lib/metal_w4a16_source.ml:1256-1283; there one
// candidate per threadgroup of columns, here candidate t is the best of columns
// t, t + 256, ... - the reduce step only needs every column covered once and
// ties resolved to the lowest index).  Four slices of threads scan a quarter
// of those columns each with several independent loads in flight, then meet in
// LDS: a single thread per candidate would walk its 192 columns of a 49152-wide
// vocabulary one load latency at a time.
constexpr int kArgmaxSlices = 4;
constexpr int kArgmaxUnroll = 16;

// Logits of a row: `low`, when not null, is the row of the products with the lo half of the activation (see
// rms_norm_split_kernel), whose sum with the hi half's is the logit; `half`, when not null, receives half(logit).
struct ArgmaxRow {
  const float *logits, *low;
  uint16_t *half;
  uint32_t n;
};

__device__ __forceinline__ ArgmaxRow argmax_row(const float *logits, uint32_t n, bool pairs, uint16_t *half_logits, uint32_t row) {
  const float *of_row = logits + (size_t)row * n * (pairs ? 2 : 1);
  return {of_row, pairs ? of_row + n : nullptr, half_logits != nullptr ? half_logits + (size_t)row * n : nullptr, n};
}

// Columns t + 256 slice, then every 1024th; index 0xffffffff: there are none.
__device__ __forceinline__ Candidate argmax_scan(const ArgmaxRow &row, uint32_t t, uint32_t slice) {
  float best_value = -3.402823466e+38f;
  uint32_t best_index = 0;
  bool found = false;
  // columns are visited in increasing order, so `>` alone keeps the lowest index among equals
  auto take = [&](uint32_t col, float value) __attribute__((always_inline)) {
    if (found && !(value > best_value)) return;
    best_value = value;
    best_index = col;
    found = true;
  };
  constexpr uint32_t step = 256 * kArgmaxSlices;
  uint32_t col = t + 256 * slice;
  for (; col < row.n && row.n - col > (kArgmaxUnroll - 1) * step; col += kArgmaxUnroll * step) {
    float value[kArgmaxUnroll], low[kArgmaxUnroll];
#pragma unroll
    for (int u = 0; u < kArgmaxUnroll; ++u) {
      value[u] = row.logits[col + u * step];
      low[u] = row.low != nullptr ? row.low[col + u * step] : 0.0f;
    }
#pragma unroll
    for (int u = 0; u < kArgmaxUnroll; ++u) {
      value[u] += low[u];
      if (row.half != nullptr) row.half[col + u * step] = float_to_half_bits(value[u]);
    }
#pragma unroll
    for (int u = 0; u < kArgmaxUnroll; ++u) take(col + u * step, value[u]);
  }
  for (; col < row.n; col += step) {
    const float value = row.logits[col] + (row.low != nullptr ? row.low[col] : 0.0f);
    if (row.half != nullptr) row.half[col] = float_to_half_bits(value);
    take(col, value);
  }
  return {best_value, found ? best_index : 0xffffffffu};
}

// Candidate t from its slices (`stride` apart).
__device__ __forceinline__ Candidate argmax_join(const Candidate *slices, uint32_t stride) {
  Candidate best = slices[0];
#pragma unroll
  for (int other = 1; other < kArgmaxSlices; ++other) {
    const Candidate c = slices[other * stride];
    if (c.index != 0xffffffffu && (best.index == 0xffffffffu || better(c.value, c.index, best.value, best.index))) best = c;
  }
  // a candidate with no column at all (n <= t): the reference's initial (lowest float, 0)
  if (best.index == 0xffffffffu) best = {-3.402823466e+38f, 0};
  return best;
}

// The best of 256 candidates by one wave, in the order of the reference's tree (lib/metal_w4a16_source.ml:1287-1315): lane l
// holds candidates l, l + 64, l + 128 and l + 192.  Lane 0 ends with it.
__device__ __forceinline__ Candidate argmax_tree(Candidate (&c)[4]) {
  auto keep = [](Candidate &mine, const Candidate &other) __attribute__((always_inline)) {
    if (better(other.value, other.index, mine.value, mine.index)) mine = other;
  };
  keep(c[0], c[2]);
  keep(c[1], c[3]);
  keep(c[0], c[1]);
#pragma unroll
  for (int width = 32; width > 0; width >>= 1) {
    const Candidate other = {__shfl_down(c[0].value, width, 64), (uint32_t)__shfl_down((int)c[0].index, width, 64)};
    keep(c[0], other);
  }
  return c[0];
}

// A workgroup owns kArgmaxGroup candidates of a row: a row of 49152 pairs is 393 KB, which one CU takes 5 us to read.
constexpr uint32_t kArgmaxGroup = 16;

__global__ __launch_bounds__(kArgmaxGroup * kArgmaxSlices) void argmax_candidates_kernel(const float *logits, Candidate *candidates,
                                                                                        uint32_t n, bool pairs, uint16_t *half_logits) {
  __shared__ Candidate slices[kArgmaxGroup * kArgmaxSlices];
  const uint32_t row = blockIdx.x, within = threadIdx.x % kArgmaxGroup, t = blockIdx.y * kArgmaxGroup + within;
  slices[threadIdx.x] = argmax_scan(argmax_row(logits, n, pairs, half_logits, row), t, threadIdx.x / kArgmaxGroup);
  __syncthreads();
  if (threadIdx.x < kArgmaxGroup) candidates[(size_t)row * 256 + t] = argmax_join(slices + within, kArgmaxGroup);
}

// lib/metal_w4a16_source.ml:1287-1315
__global__ __launch_bounds__(64) void argmax_reduce_kernel(const Candidate *candidates, uint32_t *token_ids) {
  Candidate c[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) c[j] = candidates[(size_t)blockIdx.x * 256 + threadIdx.x + 64 * j];
  const Candidate best = argmax_tree(c);
  if (threadIdx.x == 0) token_ids[blockIdx.x] = best.index;
}

// Both steps of a row by one workgroup.
__global__ __launch_bounds__(256 * kArgmaxSlices) void argmax_rows_kernel(const float *logits, uint32_t *token_ids, uint32_t n,
                                                                         bool pairs, uint16_t *half_logits) {
  __shared__ Candidate slices[kArgmaxSlices * 256];
  slices[threadIdx.x] = argmax_scan(argmax_row(logits, n, pairs, half_logits, blockIdx.x), threadIdx.x & 255, threadIdx.x >> 8);
  __syncthreads();
  if (threadIdx.x >= 64) return;
  Candidate c[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) c[j] = argmax_join(slices + threadIdx.x + 64 * j, 256);
  const Candidate best = argmax_tree(c);
  if (threadIdx.x == 0) token_ids[blockIdx.x] = best.index;
}

}  // namespace

// 16-byte requests of whole rows that fit a wave's registers.
static bool vector_rows(const RmsNormArgs &a) {
  return !a.input_f32 && a.width % 8 == 0 && a.width <= 64 * 8 * kRmsVectors &&
         ((reinterpret_cast<uintptr_t>(a.input) | reinterpret_cast<uintptr_t>(a.weight) | reinterpret_cast<uintptr_t>(a.output)) & 15) == 0;
}

hipError_t launch_rms_norm(const RmsNormArgs &a, hipStream_t stream) {
  const dim3 grid((a.rows + kRowWaves - 1) / kRowWaves), block(kRowWaves * 64);
  if (a.input_f32) {
    const float *in = static_cast<const float *>(a.input);
    if (a.weight_first)
      hipLaunchKernelGGL((rms_norm_kernel<float, true>), grid, block, 0, stream, in, a.weight, a.output, a.rows,
                         a.width, a.epsilon);
    else
      hipLaunchKernelGGL((rms_norm_kernel<float, false>), grid, block, 0, stream, in, a.weight, a.output,
                         a.rows, a.width, a.epsilon);
  } else {
    const uint16_t *in = static_cast<const uint16_t *>(a.input);
    if (vector_rows(a)) {
      if (a.weight_first)
        hipLaunchKernelGGL((rms_norm_f16_rows_kernel<true>), grid, block, 0, stream, in, a.weight, a.output, a.rows,
                           a.width, a.epsilon);
      else
        hipLaunchKernelGGL((rms_norm_f16_rows_kernel<false>), grid, block, 0, stream, in, a.weight, a.output, a.rows,
                           a.width, a.epsilon);
      return hipGetLastError();
    }
    if (a.weight_first)
      hipLaunchKernelGGL((rms_norm_kernel<uint16_t, true>), grid, block, 0, stream, in, a.weight, a.output,
                         a.rows, a.width, a.epsilon);
    else
      hipLaunchKernelGGL((rms_norm_kernel<uint16_t, false>), grid, block, 0, stream, in, a.weight, a.output,
                         a.rows, a.width, a.epsilon);
  }
  return hipGetLastError();
}

hipError_t launch_rotary_qk(const RotaryQkArgs &a, hipStream_t stream) {
  const uint32_t rows = a.batches * (a.q_heads + a.k_heads) * a.tokens;
  hipLaunchKernelGGL(rotary_qk_kernel, dim3((rows + kRowWaves - 1) / kRowWaves), dim3(kRowWaves * 64), 0,
                     stream, a);
  return hipGetLastError();
}

hipError_t launch_embedding(const EmbeddingArgs &a, hipStream_t stream) {
  const size_t count = (size_t)a.tokens * a.width;
  hipLaunchKernelGGL(embedding_kernel, dim3((uint32_t)((count + 255) / 256)), dim3(256), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_add_f16(const PointwiseArgs &a, hipStream_t stream) {
  bool same_shape = !a.left_scalar && !a.right_scalar && a.count % 8 == 0;
  for (uint32_t axis = 0; axis < a.rank && same_shape; ++axis)
    same_shape = a.left_shape[axis] == a.output_shape[axis] && a.right_shape[axis] == a.output_shape[axis];
  const auto aligned = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  if (same_shape && aligned(a.left) && aligned(a.right) && aligned(a.output)) {
    const uint32_t vectors = a.count / 8;
    hipLaunchKernelGGL(add_f16_same_shape_kernel, dim3((vectors + 255) / 256), dim3(256), 0, stream,
                       reinterpret_cast<const uint4 *>(a.left), reinterpret_cast<const uint4 *>(a.right),
                       reinterpret_cast<uint4 *>(a.output), vectors);
  } else {
    hipLaunchKernelGGL(add_f16_kernel, dim3((a.count + 255) / 256), dim3(256), 0, stream, a);
  }
  return hipGetLastError();
}

namespace {
// The per-step state of a retained decode plan, written in stream order ahead of its graph:
// the input token (given, or the previous step's output token: llmopt_chain_token_id,
// native/ocaml_metal_stubs.m:1570-1577) and the context length every sequence attends to.
__global__ void plan_state_kernel(int64_t *token, int64_t value, const int32_t *chain_from, uint32_t *past,
                                  uint32_t past_value, uint32_t past_count, uint32_t *checkpoint,
                                  uint32_t checkpoint_value) {
  if (threadIdx.x == 0 && token != nullptr) *token = chain_from != nullptr ? (int64_t)*chain_from : value;
  if (threadIdx.x == 0 && checkpoint != nullptr) *checkpoint = checkpoint_value;
  for (uint32_t i = threadIdx.x; i < past_count; i += blockDim.x) past[i] = past_value;
}

// Loads that pass the caches by (the host writes these words anew for every replay), all in one trip.
__global__ void plan_begin_kernel(const StepWords *step) {
  constexpr int WORDS = offsetof(StepWords, result) / 8;
  static_assert(offsetof(StepWords, result) == 8 * WORDS, "whole words");
  union {
    uint64_t words[WORDS];
    StepWords step;
  } s;
#pragma unroll
  for (int i = 0; i < WORDS; ++i)
    s.words[i] = __hip_atomic_load(reinterpret_cast<const uint64_t *>(step) + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  if (threadIdx.x == 0) {
    if (s.step.resident != nullptr) {
      s.step.resident[0] = s.step.resident_tag;
      s.step.resident[1] = 0;
    }
    if (s.step.token != nullptr) *s.step.token = s.step.value;
    if (s.step.checkpoint != nullptr) *s.step.checkpoint = s.step.checkpoint_value;
  }
  for (uint32_t i = threadIdx.x; i < s.step.past_count; i += blockDim.x) s.step.past[i] = s.step.past_value;
}

__global__ void plan_result_kernel(const int32_t *output, const uint32_t *failed, int32_t *host) {
  if (threadIdx.x != 0) return;
  host[0] = output != nullptr ? *output : 0;
  if (failed != nullptr) host[1] = (int32_t)*failed;
}

// *found = 1 when the range holds a NaN (not an infinity): fp16 words, or float32 words.
__global__ void nan_scan_kernel(const uint8_t *data, size_t words, bool f32, uint32_t *found) {
  bool seen = false;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < words; i += (size_t)gridDim.x * blockDim.x) {
    if (f32) {
      const uint32_t v = reinterpret_cast<const uint32_t *>(data)[i];
      seen |= (v & 0x7F800000u) == 0x7F800000u && (v & 0x007FFFFFu) != 0;
    } else {
      const uint16_t v = reinterpret_cast<const uint16_t *>(data)[i];
      seen |= (v & 0x7C00u) == 0x7C00u && (v & 0x03FFu) != 0;
    }
  }
  if (seen) *found = 1u;  // every writer stores the same value
}
}  // namespace

hipError_t launch_nan_scan(const void *data, size_t bytes, bool f32, uint32_t *found, hipStream_t stream) {
  const size_t words = bytes / (f32 ? 4 : 2);
  if (words == 0) return hipSuccess;
  const uint32_t blocks = (uint32_t)std::min<size_t>((words + 255) / 256, 2048);
  hipLaunchKernelGGL(nan_scan_kernel, dim3(blocks), dim3(256), 0, stream, static_cast<const uint8_t *>(data), words, f32,
                     found);
  return hipGetLastError();
}

hipError_t launch_plan_state(int64_t *token, int64_t value, const int32_t *chain_from, uint32_t *past,
                             uint32_t past_value, uint32_t past_count, uint32_t *checkpoint, uint32_t checkpoint_value,
                             hipStream_t stream) {
  hipLaunchKernelGGL(plan_state_kernel, dim3(1), dim3(256), 0, stream, token, value, chain_from, past, past_value,
                     past_count, checkpoint, checkpoint_value);
  return hipGetLastError();
}

hipError_t launch_plan_begin(const StepWords *step, hipStream_t stream) {
  hipLaunchKernelGGL(plan_begin_kernel, dim3(1), dim3(64), 0, stream, step);
  return hipGetLastError();
}

hipError_t launch_plan_result(const int32_t *output, const uint32_t *failed, int32_t *host, hipStream_t stream) {
  hipLaunchKernelGGL(plan_result_kernel, dim3(1), dim3(64), 0, stream, output, failed, host);
  return hipGetLastError();
}

hipError_t launch_copy_bytes(void *destination, const void *source, size_t bytes, hipStream_t stream) {
  if (bytes == 0) return hipSuccess;
  const bool vector_ok = ((reinterpret_cast<uintptr_t>(destination) | reinterpret_cast<uintptr_t>(source)) & 15) == 0;
  const size_t vectors = vector_ok ? bytes / 16 : 0;
  if (vectors > 0) {
    const size_t wanted = (vectors + 255) / 256;
    const uint32_t blocks = (uint32_t)std::min<size_t>(wanted, 8192);
    hipLaunchKernelGGL(copy_vectors_kernel, dim3(blocks), dim3(256), 0, stream,
                       static_cast<const u32x4_t *>(source), static_cast<u32x4_t *>(destination), vectors);
  }
  const size_t done = vectors * 16;
  if (done < bytes) {
    const size_t rest = bytes - done;
    const uint32_t blocks = (uint32_t)std::min<size_t>((rest + 255) / 256, 8192);
    hipLaunchKernelGGL(copy_bytes_kernel, dim3(blocks), dim3(256), 0, stream,
                       static_cast<const uint8_t *>(source) + done, static_cast<uint8_t *>(destination) + done, rest);
  }
  return hipGetLastError();
}

hipError_t launch_argmax_candidates(const float *logits, void *candidates, uint32_t rows, uint32_t n, bool pairs,
                                    uint16_t *half_logits, hipStream_t stream) {
  hipLaunchKernelGGL(argmax_candidates_kernel, dim3(rows, 256 / kArgmaxGroup), dim3(kArgmaxGroup * kArgmaxSlices), 0, stream,
                     logits, static_cast<Candidate *>(candidates), n, pairs, half_logits);
  return hipGetLastError();
}

// One workgroup a row up to 144 KB of logits, us one launch / two: 8192 3.6 / 4.2, 32768 5.1 / 5.4, 49152 6.2 / 6.2, 65536 7.2 /
// 7.0, 49152 pairs with their halves stored (behind the head's product) 21.7 / 19.7.  (A thread for every candidate and slice in
// one workgroup, then a launch that joined them over eight barriers: 5.9 at 32768, 26.8 with the head.)
constexpr uint64_t kArgmaxOneLaunchBytes = 144 << 10;

hipError_t launch_argmax(const float *logits, void *candidates, uint32_t *token_ids, uint32_t rows, uint32_t n, bool pairs,
                         uint16_t *half_logits, hipStream_t stream) {
  if ((uint64_t)n * (pairs ? 8 : 4) <= kArgmaxOneLaunchBytes) {
    hipLaunchKernelGGL(argmax_rows_kernel, dim3(rows), dim3(256 * kArgmaxSlices), 0, stream, logits, token_ids, n, pairs,
                       half_logits);
    return hipGetLastError();
  }
  if (hipError_t status = launch_argmax_candidates(logits, candidates, rows, n, pairs, half_logits, stream)) return status;
  return launch_argmax_reduce(candidates, token_ids, rows, stream);
}

hipError_t launch_rms_norm_split(const RmsNormArgs &a, hipStream_t stream) {
  const dim3 grid((a.rows + kRowWaves - 1) / kRowWaves), block(kRowWaves * 64);
  if (vector_rows(a))
    hipLaunchKernelGGL((rms_norm_f16_rows_kernel<true, true>), grid, block, 0, stream, static_cast<const uint16_t *>(a.input),
                       a.weight, a.output, a.rows, a.width, a.epsilon);
  else if (a.input_f32)
    hipLaunchKernelGGL(rms_norm_split_kernel<float>, grid, block, 0, stream, static_cast<const float *>(a.input),
                       a.weight, a.output, a.rows, a.width, a.epsilon);
  else
    hipLaunchKernelGGL(rms_norm_split_kernel<uint16_t>, grid, block, 0, stream,
                       static_cast<const uint16_t *>(a.input), a.weight, a.output, a.rows, a.width, a.epsilon);
  return hipGetLastError();
}

hipError_t launch_argmax_reduce(const void *candidates, uint32_t *token_ids, uint32_t rows, hipStream_t stream) {
  hipLaunchKernelGGL(argmax_reduce_kernel, dim3(rows), dim3(64), 0, stream,
                     static_cast<const Candidate *>(candidates), token_ids);
  return hipGetLastError();
}

}  // namespace llmopt
