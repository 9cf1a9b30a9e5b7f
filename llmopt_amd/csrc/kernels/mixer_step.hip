// One token through window attention and the gated delta rule side by side: one launch for both mixers, two where the
// keys' shares are merged apart (joins_shares).
//
// Alone, each mixer of a token is a few workgroups that wait for memory (7.2 us attention, 2.2 its merge, 13.8 a workgroup
// per head of the delta rule, at 16 heads of 64 and 8 of 128 x 128): together they take as long as the longer one.
//  * mixer_step_kernel: the first workgroups take 32 value columns of a delta-rule head each, the others a share of a
//    key / value head's keys (chunk_decode.h).  A head's state passes through registers, a row of 32 columns by eight
//    lanes; every workgroup of a head forms the head's decays and unit vectors for itself.  The output's norm needs all
//    columns: the workgroups leave their values and sums of squares, and the last of a head to arrive divides the row by
//    its root mean square.
// Measured at those sizes, four layers: a prompt of 64 tokens and 24 decoded ones 6226 us with a launch for every part,
// 5080 with both mixers in one launch and a finishing one (3.9 us of 34 a layer), 4530 without that.
#include <algorithm>

#include "chunk_decode.h"
#include "dense.h"
#include "dense_common.h"
#include "kernels_internal.h"

namespace llmopt {
namespace {

constexpr int kThreads = 512, kWaves = kThreads / 64;
constexpr uint32_t kColumns = 32, kRowsAPass = kThreads / 8;
constexpr uint32_t kMaxRank = 128;
constexpr float kUnitEpsilon = 1e-6f;

struct DeltaStepLds {
  float key[kDeltaMaxWidth], query[kDeltaMaxWidth], decay[kDeltaMaxWidth], gate[kColumns];
  float read[kWaves][kColumns], out[kWaves][kColumns], written[kColumns];
  float product;
};

__device__ __forceinline__ float bf16_at(const uint16_t *p, size_t i) { return (float)reinterpret_cast<const __bf16 *>(p)[i]; }

// R: passes of 64 rows over the state (dim <= 64 R).  A wave issues an instruction every four or five cycles and these waves have
// nothing else to do: what counts is how many there are and how many trips lie behind one another.  With the decays' exponentials one
// thread a row (five rows one after the other in one lane of sixteen), sums between lanes without LDS and the parts' squares asked
// for together: 9.1 to 9.8 us -> 7.8 to 8.4 the launch, a token of four layers 161.6 -> 153.6.
template <int R>
__device__ __forceinline__ void delta_columns(const DeltaArgs &a, uint32_t head, uint32_t part, DeltaStepLds &lds,
                                              float *squares, uint32_t *counter) {
  constexpr int PASSES = 2 * R;  // of 32 rows over those of the decays' low-rank product; the gate's are kColumns rows, one pass
  static_assert(kThreads / 16 == kColumns, "a pass takes the rows of the gate");
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const uint32_t group = head / (a.heads / a.kv_heads), parts = a.vdim / kColumns;
  const uint32_t column = part * kColumns + (tid & 7) * 4, first = tid >> 3;
  const bool fresh = a.step[kStatePosition] == 0;
  float *state = a.state + ((size_t)a.step[kStateSlot] * a.heads + head) * a.dim * a.vdim + column;

  // Asked for in the order in which it is needed, all before the first use.
  const float *queries = a.row + (size_t)group * a.dim, *keys = queries + (size_t)a.kv_heads * a.dim;
  float q[R], k[R];  // 64 components each: wave 0 takes the query's length, wave 1 the key's, wave 2 their product
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const uint32_t c = lane + 64 * i;
    q[i] = wave < 3 && wave != 1 && c < a.dim ? queries[c] : 0.0f;
    k[i] = wave < 3 && wave != 0 && c < a.dim ? keys[c] : 0.0f;
  }
  // sixteen lanes a row of the low-rank products, eight values each
  const uint32_t piece = (tid & 15) * 8, row = tid >> 4;
  const uint32_t decay_piece = min(piece, a.decay_rank - 8), gate_piece = min(piece, a.gate_rank - 8);
  bf16x8 weights[PASSES + 1];
#pragma unroll
  for (int i = 0; i < PASSES; ++i)
    weights[i] = *reinterpret_cast<const bf16x8 *>(a.w_decay + ((size_t)head * a.dim + min(row + 32 * i, a.dim - 1)) * a.decay_rank + decay_piece);
  weights[PASSES] = *reinterpret_cast<const bf16x8 *>(a.w_gate + ((size_t)head * a.vdim + part * kColumns + row) * a.gate_rank + gate_piece);
  f32x4 inputs[2][2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    inputs[0][h] = *reinterpret_cast<const f32x4 *>(a.decay_in + decay_piece + 4 * h);
    inputs[1][h] = *reinterpret_cast<const f32x4 *>(a.gate_in + gate_piece + 4 * h);
  }
  const float dt_bias = bf16_at(a.dt_bias, (size_t)head * a.dim + min((uint32_t)tid, a.dim - 1));
  const float log_rate = bf16_at(a.a_log, head), raw_beta = a.row_beta[head];
  const uint32_t own = part * kColumns + (lane & (kColumns - 1));  // the column of wave 0's lane
  const float own_norm = bf16_at(a.norm, own), own_value = a.row[2 * (size_t)a.kv_heads * a.dim + (size_t)head * a.vdim + own];
  f32x4 s[R];
#pragma unroll
  for (int i = 0; i < R; ++i) s[i] = *reinterpret_cast<const f32x4 *>(state + (size_t)min(first + kRowsAPass * i, a.dim - 1) * a.vdim);

  if (wave < 3) {
    float qq = 0.0f, kk = 0.0f, qk = 0.0f;
#pragma unroll
    for (int i = 0; i < R; ++i) {
      qq += q[i] * q[i];
      kk += k[i] * k[i];
      qk += q[i] * k[i];
    }
    const float q_scale = wave == 1 ? 0.0f : 1.0f / sqrtf(wave_sum(qq) + kUnitEpsilon) / sqrtf((float)a.dim);
    const float k_scale = wave == 0 ? 0.0f : 1.0f / sqrtf(wave_sum(kk) + kUnitEpsilon);
    if (wave == 2) {
      qk = wave_sum(qk);
      if (lane == 0) lds.product = qk * q_scale * k_scale;
    } else {
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const uint32_t c = lane + 64 * i;
        if (c < a.dim) (wave == 0 ? lds.query : lds.key)[c] = wave == 0 ? q[i] * q_scale : k[i] * k_scale;
      }
    }
  }
  // the low-rank sums, then one thread a row for what becomes of them
#pragma unroll
  for (int i = 0; i < PASSES + 1; ++i) {
    const bool gates = i == PASSES;
    float sum = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) sum = fmaf((float)weights[i][e], inputs[gates][e / 4][e % 4], sum);
    sum = row_sum(piece < (gates ? a.gate_rank : a.decay_rank) ? sum : 0.0f);
    const uint32_t r = row + 32 * i;
    if ((tid & 15) == 0 && (gates || r < a.dim)) (gates ? lds.gate[row] : lds.decay[r]) = sum;
  }
  __syncthreads();
  if ((uint32_t)tid < a.dim) lds.decay[tid] = expf(-expf(log_rate) * softplus_f32(lds.decay[tid] + dt_bias));
  __syncthreads();

  f32x4 from_key = 0.0f, from_query = 0.0f;
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const uint32_t r = first + kRowsAPass * i;
    const bool there = r < a.dim;
    const uint32_t at = there ? r : a.dim - 1;
    s[i] = fresh || !there ? f32x4{0.0f, 0.0f, 0.0f, 0.0f} : s[i] * lds.decay[at];
    from_key += s[i] * lds.key[at];
    from_query += s[i] * lds.query[at];
  }
  // the eight rows of a wave, then the waves
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    from_key[e] += dpp_f32<0x128>(from_key[e]);  // row_ror 8
    from_query[e] += dpp_f32<0x128>(from_query[e]);
    from_key[e] = add_32_away(add_16_away(from_key[e]));
    from_query[e] = add_32_away(add_16_away(from_query[e]));
  }
  if (lane < 8) {
    *reinterpret_cast<f32x4 *>(&lds.read[wave][lane * 4]) = from_key;
    *reinterpret_cast<f32x4 *>(&lds.out[wave][lane * 4]) = from_query;
  }
  __syncthreads();
  if (wave == 0) {
    float out = 0.0f;
    if (lane < (int)kColumns) {
      float read = 0.0f;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        read += lds.read[w][lane];
        out += lds.out[w][lane];
      }
      const float u = sigmoid_f32(raw_beta) * (own_value - read);
      lds.written[lane] = u;
      out = fmaf(lds.product, u, out);
      hand_over(a.out_row + (size_t)head * a.vdim + own, out * own_norm * sigmoid_f32(lds.gate[lane]) * a.out_scale);
    }
    const float square = wave_sum(out * out);
    if (lane == 0) hand_over(squares + head * parts + part, square);
  }
  __syncthreads();
  const f32x4 u = *reinterpret_cast<const f32x4 *>(&lds.written[(tid & 7) * 4]);
  auto store_state = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const uint32_t r = first + kRowsAPass * i;
      if (r < a.dim) *reinterpret_cast<f32x4 *>(state + (size_t)r * a.vdim) = s[i] + lds.key[r] * u;
    }
  };
  if (wave != 0) return store_state();
  // the last part of a head to arrive divides the head's row by its root mean square, all in this wave (which stores its share of
  // the state behind that: loads behind stores wait for them)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  bool last = false;
  if (lane == 0) last = last_to_arrive(counter, parts - 1);
  if (__shfl((int)last, 0, 64) != 0) {
    constexpr int MOST = kDeltaMaxWidth / kColumns;
    float *out = a.out_row + (size_t)head * a.vdim, value[kDeltaMaxWidth / 64], square[MOST], total = 0.0f;
#pragma unroll
    for (int i = 0; i < (int)kDeltaMaxWidth / 64; ++i) value[i] = lane + 64 * i < a.vdim ? handed_over(out + lane + 64 * i) : 0.0f;
#pragma unroll
    for (int p = 0; p < MOST; ++p) square[p] = handed_over(squares + head * parts + min((uint32_t)p, parts - 1));
#pragma unroll
    for (int p = 0; p < MOST; ++p) total += p < parts ? square[p] : 0.0f;
    const float inverse = 1.0f / sqrtf(total / (float)a.vdim + a.epsilon);
#pragma unroll
    for (int i = 0; i < (int)kDeltaMaxWidth / 64; ++i)
      if (lane + 64 * i < a.vdim) out[lane + 64 * i] = value[i] * inverse;
  }
  store_state();
}

template <int ND, int NE>
constexpr int attention_lds_bytes() { return decode_lds_floats<__bf16, NE>() * 4 + raw_row_lds_bytes<__bf16, ND, NE>(); }

template <int ND, int NE, int R, bool JOIN, bool FULL>
__global__ __launch_bounds__(kThreads) void mixer_step_kernel(ChunkAttentionArgs a, DeltaArgs d, uint32_t splits, float *squares, uint32_t *counters) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const uint32_t parts = d.vdim / kColumns, delta_blocks = d.heads * parts;
  if (blockIdx.x < delta_blocks) {
    delta_columns<R>(d, blockIdx.x / parts, blockIdx.x % parts, *reinterpret_cast<DeltaStepLds *>(lds), squares,
                     counters + blockIdx.x / parts);
    return;
  }
  if (threadIdx.x >= 256) return;  // (barriers count the waves that are still there)
  const uint32_t share = blockIdx.x - delta_blocks;
  chunk_decode<__bf16, ND, NE, true, JOIN, FULL>(a, splits, share % a.kv_heads, share / a.kv_heads, lds, counters + d.heads);
}

__global__ __launch_bounds__(256) void mixer_merge_kernel(ChunkAttentionArgs a, uint32_t splits) {
  extern __shared__ __attribute__((aligned(16))) float shared[];
  chunk_merge<__bf16>(a, splits, blockIdx.x, shared);
}

template <int ND, int NE, int R>
hipError_t run(const ChunkAttentionArgs &a, const DeltaArgs &d, float *squares, hipStream_t stream) {
  constexpr int bytes = std::max<int>(attention_lds_bytes<ND, NE>(), (int)sizeof(DeltaStepLds));
  static_assert(bytes <= 64 * 1024, "no raised limit");
  const uint32_t splits = decode_splits(a), blocks = d.heads * (d.vdim / kColumns) + a.kv_heads * splits;
  ChunkAttentionArgs own = a;  // (the attention's counters lie behind the delta rule's)
  own.counter_count -= d.heads;
  const bool joins = joins_shares(own);
  const auto kernel = full_heads<__bf16, ND, NE>(a)
                          ? (joins ? mixer_step_kernel<ND, NE, R, true, true> : mixer_step_kernel<ND, NE, R, false, true>)
                          : (joins ? mixer_step_kernel<ND, NE, R, true, false> : mixer_step_kernel<ND, NE, R, false, false>);
  kernel<<<blocks, kThreads, bytes, stream>>>(a, d, splits, squares, a.counters);
  if (hipError_t status = hipGetLastError()) return status;
  if (splits > 1 && !joins) mixer_merge_kernel<<<a.heads, 256, splits * 8, stream>>>(a, splits);
  return hipGetLastError();
}

template <int ND, int NE>
hipError_t pick_rows(const ChunkAttentionArgs &a, const DeltaArgs &d, float *squares, hipStream_t stream) {
  if (d.dim <= 128) return run<ND, NE, 2>(a, d, squares, stream);
  return run<ND, NE, 4>(a, d, squares, stream);
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace

// The wide loads' conditions: whole sixteen-byte pieces of every low-rank row and of its inputs, whole parts of 32 value
// columns; heads of attention up to 128 values (wider ones hold too many registers beside the other half).
bool mixer_step_ok(const ChunkAttentionArgs &a, const DeltaArgs &d) {
  return !a.f32 && a.m == 1 && d.m == 1 && a.row != nullptr && a.counters != nullptr && d.heads <= a.counter_count && a.dim <= 128 && a.vdim > 32 && a.vdim <= 128 &&
         chunk_attention_ok(a) && d.dim <= kDeltaMaxWidth && d.vdim <= kDeltaMaxWidth && d.vdim % kColumns == 0 &&
         d.decay_rank >= 8 && d.gate_rank >= 8 && d.decay_rank <= kMaxRank && d.gate_rank <= kMaxRank &&
         (d.decay_rank | d.gate_rank) % 8 == 0 && aligned16(d.decay_in) && aligned16(d.gate_in) && aligned16(d.w_decay) &&
         aligned16(d.w_gate) && aligned16(d.state);
}

size_t mixer_step_squares(const DeltaArgs &d) { return (size_t)d.heads * (d.vdim / kColumns) * sizeof(float); }

hipError_t launch_mixer_step(const ChunkAttentionArgs &a, const DeltaArgs &d, float *squares, hipStream_t stream) {
  if (a.dim <= 64) return a.vdim <= 64 ? pick_rows<2, 4>(a, d, squares, stream) : pick_rows<2, 8>(a, d, squares, stream);
  return a.vdim <= 64 ? pick_rows<4, 4>(a, d, squares, stream) : pick_rows<4, 8>(a, d, squares, stream);
}

}  // namespace llmopt
