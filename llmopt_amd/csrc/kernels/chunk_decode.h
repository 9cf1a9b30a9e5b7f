// Device code of one token's chunk or window attention (chunk_attention.hip, mixer_step.hip): a workgroup's share of the
// keys, the merge of the shares, and the norm and rotation of heads.
#pragma once

#include "chunk_join_rule.h"
#include "dense.h"
#include "dense_common.h"

namespace llmopt {

constexpr uint32_t kSplitKeys = 128;
constexpr float kLog2e = 1.4426950408889634f;

// The first position that `position` sees; never falls from one position to the next.
__device__ __forceinline__ uint32_t first_seen(uint32_t position, const ChunkCache &cache) {
  if (cache.span == 0) return 0;
  if (cache.sliding) return position + 1 > cache.span ? position + 1 - cache.span : 0;
  return position - position % cache.span;
}

// Values of four keys (rows of the stage) at the lane's column: what the V^T operand takes.  bf16: the
// transposing LDS read - in a group of 16 lanes, lane 4 q + c receives element c of the 8-byte pieces named
// by lanes q, 4 + q, 8 + q and 12 + q, so lane 4 e + q names (key e, columns 4 q ..).
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 *lds_piece_t;
__device__ __forceinline__ bf16x4 four_keys(const __bf16 *stage, int stride, int lane) {
  const __bf16 *piece = stage + ((lane & 15) >> 2) * stride + (lane & 3) * 4;
  return __builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_piece_t)piece));
}
__device__ __forceinline__ f32x4 four_keys(const float *stage, int stride, int lane) {
  f32x4 v;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = stage[i * stride + (lane & 15)];
  return v;
}

__device__ __forceinline__ float exp2_raw(float x) { return __builtin_amdgcn_exp2f(x); }

template <typename T, int NE>
constexpr int value_stride() { return NE * 16 + 32 / (int)sizeof(T); }

// One token: the query heads of one key / value head are the operand columns (16 at a time), a wave takes 32
// keys of the workgroup's 128; all keys and values of a split are requested before the first is used.  The
// values pass through a wave's own LDS rows on the way to their transposed operand.  Partial results
// [heads][splits][vdim + 2] (weighted sum, maximum, total), or the output when there is one split.
template <typename T, int NE>
constexpr int decode_lds_floats() {
  return 4 * 32 * value_stride<T, NE>() * (int)sizeof(T) / 4 + 2 * 4 * 16;
}

// Cosine and sine of every rotated pair at one position.
struct Turn {
  float cosine, sine;
};
__device__ __forceinline__ void fill_turns(const HeadRotation &r, uint32_t position, Turn *turns) {
  for (uint32_t c = threadIdx.x; c < r.dims / 2; c += 256) turn(position, r.frequencies[c], turns[c].cosine, turns[c].sine);
}

// Norm and rotation of head vectors, a wave a vector, lane l holding components l + 64 i.
template <int PARTS>
struct HeadVector {
  float v[PARTS];
  // exchange(v, partner, half): every rotated component's partner, c + half or c - half.
  template <typename Exchange>
  __device__ __forceinline__ void norm_and_rotate(const HeadRotation &r, const uint16_t *norm, uint32_t dim,
                                                  const Turn *turns, int lane, Exchange exchange) {
    float weight[PARTS];
    norm_weights(norm, dim, lane, weight);
    normalise(r, weight, dim);
    rotate(r, turns, lane, exchange);
  }
  static __device__ __forceinline__ void norm_weights(const uint16_t *norm, uint32_t dim, int lane, float (&weight)[PARTS]) {
#pragma unroll
    for (int i = 0; i < PARTS; ++i) {
      const uint32_t c = lane + 64 * i;
      weight[i] = c < dim ? (float)reinterpret_cast<const __bf16 *>(norm)[c] : 0.0f;
    }
  }
  __device__ __forceinline__ void normalise(const HeadRotation &r, const float (&weight)[PARTS], uint32_t dim) {
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < PARTS; ++i) sum += v[i] * v[i];
    const float inverse = 1.0f / sqrtf(wave_sum(sum) / (float)dim + r.epsilon);
#pragma unroll
    for (int i = 0; i < PARTS; ++i) v[i] *= inverse * weight[i];
  }
  template <typename Exchange>
  __device__ __forceinline__ void rotate(const HeadRotation &r, const Turn *turns, int lane, Exchange exchange) {
    float partner[PARTS];
    const uint32_t half = r.dims / 2;
    exchange(v, partner, half);
#pragma unroll
    for (int i = 0; i < PARTS; ++i) {
      const uint32_t c = lane + 64 * i;
      if (c >= r.dims) continue;
      const Turn t = turns[c < half ? c : c - half];
      v[i] = c < half ? v[i] * t.cosine - partner[i] * t.sine : v[i] * t.cosine + partner[i] * t.sine;
    }
  }
};

// The partner of every rotated component through `row`, floats of the wave's own in LDS.
template <int PARTS>
struct ThroughLds {
  float *row;
  uint32_t dims;
  int lane;
  __device__ __forceinline__ void operator()(const float (&v)[PARTS], float (&partner)[PARTS], uint32_t half) const {
#pragma unroll
    for (int i = 0; i < PARTS; ++i) row[lane + 64 * i] = v[i];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < PARTS; ++i) {
      const uint32_t c = lane + 64 * i;
      partner[i] = c < dims ? row[c < half ? c + half : c - half] : 0.0f;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read before the row is written again
    __builtin_amdgcn_wave_barrier();
  }
};

// LDS of a decode workgroup that starts from a raw row: queries [16][ND * 32 + pad], the own key, the own
// value, a float row for every wave, the position's turns.
template <typename T, int ND, int NE>
constexpr int raw_row_lds_bytes() {
  return (17 * (ND * 32 + 16 / (int)sizeof(T)) + NE * 16) * (int)sizeof(T) + 4 * (ND <= 2 ? 64 : ND * 32) * 4 +
         ND * 16 * (int)sizeof(Turn);
}

__device__ __forceinline__ void hand_over(float *to, float v) {
  __hip_atomic_store(to, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float handed_over(const float *from) {
  return __hip_atomic_load(from, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Whether the caller's stores and those of `others` more arrivals are all there.  The caller has waited for its own.
__device__ __forceinline__ bool last_to_arrive(uint32_t *counter, uint32_t others) {
  const bool last = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == others;
  if (last) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return last;
}

template <typename T>
__device__ __forceinline__ void store_attention(const ChunkAttentionArgs &a, uint32_t head, uint32_t c, float v) {
  if (a.out_row) a.out_row[head * a.vdim + c] = v * a.out_scale;
  else static_cast<T *>(a.out)[head * a.vdim + c] = (T)(v * a.out_scale);
}

// Up to SHARES shares in one trip and without a barrier: every thread forms its head's weights for itself.
template <typename T, uint32_t SHARES>
__device__ __forceinline__ void join_in_registers(const ChunkAttentionArgs &a, uint32_t splits, uint32_t group, uint32_t live, const float *partials) {
  const uint32_t per = a.heads / a.kv_heads, stride = a.vdim + 2;
  for (uint32_t i = threadIdx.x; i < per * a.vdim; i += 256) {
    const uint32_t h = i / a.vdim, c = i % a.vdim;
    const float *shares = partials + (size_t)h * splits * stride;
    float v[SHARES], best[SHARES], total[SHARES];
#pragma unroll
    for (uint32_t s = 0; s < SHARES; ++s) {
      const float *share = shares + min(s, live - 1) * stride;
      v[s] = handed_over(share + c);
      best[s] = handed_over(share + a.vdim);
      total[s] = handed_over(share + a.vdim + 1);
    }
    const float sink = a.sink ? (float)reinterpret_cast<const __bf16 *>(a.sink)[group * per + h] * kLog2e : -INFINITY;
    float top = sink;
#pragma unroll
    for (uint32_t s = 0; s < SHARES; ++s) top = fmaxf(top, best[s]);  // (the last one again behind the last)
    float denominator = exp2_raw(sink - top), sum = 0.0f;
#pragma unroll
    for (uint32_t s = 0; s < SHARES; ++s)
      if (s < live) {
        const float weight = exp2_raw(best[s] - top);
        denominator = fmaf(total[s], weight, denominator);
        sum = fmaf(v[s], weight, sum);
      }
    store_attention<T>(a, group * per + h, c, sum / denominator);
  }
}

// The last workgroup of a key / value head to arrive merges the head's shares itself: the sums and their order are
// chunk_merge's.  lds: two words a share and head, and one a head.
template <typename T>
__device__ __forceinline__ void join_shares(const ChunkAttentionArgs &a, uint32_t splits, uint32_t group, uint32_t live, uint32_t *counter,
                                            char *lds) {
  const uint32_t per = a.heads / a.kv_heads, stride = a.vdim + 2, tid = threadIdx.x;
  uint32_t *flag = reinterpret_cast<uint32_t *>(lds);
  float *denominators = reinterpret_cast<float *>(lds) + 1, *weights = denominators + per, *totals = weights + per * live;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();  // the stores of every wave are there
  if (tid == 0) *flag = last_to_arrive(counter, live - 1) ? 1u : 0u;
  __syncthreads();
  if (*flag == 0) return;
  const float *partials = static_cast<const float *>(a.workspace) + (size_t)group * per * splits * stride;
  if (live <= 8) return join_in_registers<T, 8>(a, splits, group, live, partials);
  if (live <= 16) return join_in_registers<T, 16>(a, splits, group, live, partials);
  for (uint32_t i = tid; i < per * live; i += 256) {
    const float *own = partials + ((size_t)(i / live) * splits + i % live) * stride + a.vdim;
    const float best = handed_over(own), total = handed_over(own + 1);
    weights[i] = best;
    totals[i] = total;
  }
  __syncthreads();
  for (uint32_t h = tid; h < per; h += 256) {
    const float sink = a.sink ? (float)reinterpret_cast<const __bf16 *>(a.sink)[group * per + h] * kLog2e : -INFINITY;
    float top = sink;
    for (uint32_t s = 0; s < live; ++s) top = fmaxf(top, weights[h * live + s]);
    float denominator = exp2_raw(sink - top);
    for (uint32_t s = 0; s < live; ++s) {
      const float weight = exp2_raw(weights[h * live + s] - top);
      weights[h * live + s] = weight;
      denominator = fmaf(totals[h * live + s], weight, denominator);
    }
    denominators[h] = denominator;
  }
  __syncthreads();
  constexpr uint32_t AHEAD = 8;
  for (uint32_t i = tid; i < per * a.vdim; i += 256) {
    const uint32_t h = i / a.vdim, c = i % a.vdim;
    const float *values = partials + (size_t)h * splits * stride + c;
    float sum = 0.0f;
    for (uint32_t s0 = 0; s0 < live; s0 += AHEAD) {
      float v[AHEAD];
#pragma unroll
      for (uint32_t s = 0; s < AHEAD; ++s) v[s] = handed_over(values + (size_t)min(s0 + s, live - 1) * stride);
#pragma unroll
      for (uint32_t s = 0; s < AHEAD; ++s)
        if (s0 + s < live) sum = fmaf(v[s], weights[h * live + s0 + s], sum);
    }
    store_attention<T>(a, group * per + h, c, sum / denominators[h]);
  }
}

// The work of one workgroup of 256 threads; lds: decode_lds_floats (and raw_row_lds_bytes behind them).  JOIN: the last
// workgroup of a key / value head (counters: one each) joins its shares; else they are a launch of their own.
// FULL: heads of just ND * 32 and NE * 16 bf16 values.  The code for partial pieces stands behind every load, and is fetched from
// memory to be jumped over.  A token of four layers of 16 heads over 4 of 64 beside the delta rule: 146.9 us, with a raw row's vectors
// asked for ahead of the keys 145.2, without that code too 142.9; of two attention layers among four 144.9, 144.2, 142.5.  Calls alone,
// 16 heads over 4 with one live share, with / without that code: rows of 64 x 64 4.1 / 3.6 us, 256 x 32 4.9 / 4.5, raw rows of 64 x 64
// 5.7 / 5.0, 256 x 256 13.1 / 11.8; every pair of widths, also with sixteen live shares and with 32 heads over 8, is 1 to 16 % shorter.
template <typename T, int ND, int NE, bool RAW, bool JOIN, bool FULL>
__device__ __forceinline__ void chunk_decode(const ChunkAttentionArgs &a, uint32_t splits, uint32_t group, uint32_t split,
                                             char *lds, uint32_t *counters) {
  constexpr int EP = NE * 16, SV = value_stride<T, NE>(), V_PIECES = EP / 8;
  const uint32_t position = a.state[kStatePosition], slot = a.state[kStateSlot];
  const uint32_t per = a.heads / a.kv_heads, dim = FULL ? ND * 32 : a.dim, vdim = FULL ? NE * 16 : a.vdim;
  const bool vec = FULL || (dim % 8 == 0 && vdim % 8 == 0);
  const uint32_t begin = first_seen(position, a.cache) + split * kSplitKeys;
  if (begin > position) return;
  const uint32_t live = min(splits, (position - first_seen(position, a.cache)) / kSplitKeys + 1);
  const bool alone = splits == 1 || (JOIN && live == 1);
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, column = lane & 15, quad = lane >> 4;
  // a wave's own rows: the values [32][SV], then its sums [16][EP] in their place
  constexpr int OWN = 32 * SV * (int)sizeof(T);
  static_assert(16 * EP * 4 <= OWN, "the sums fit the values' place");
  T *lds_v = reinterpret_cast<T *>(lds + wave * OWN);
  float *lds_top = reinterpret_cast<float *>(lds + 4 * OWN), *lds_total = lds_top + 4 * 16;  // [4][16] each
  const size_t ring = ((size_t)slot * a.kv_heads + group) * a.cache.capacity;
  const T *cache_k = static_cast<const T *>(a.cache.keys) + ring * dim;
  const T *cache_v = static_cast<const T *>(a.cache.values) + ring * vdim;
  const uint32_t wave_begin = begin + wave * 32;

  // A raw row's first vectors of each wave, their norms and the own value are asked for ahead of the keys: behind the keys and the
  // position's turns they were two trips of their own.
  constexpr int PARTS = ND <= 2 ? 1 : ND / 2, FIRST = 2;
  HeadVector<PARTS> first[FIRST];
  float first_weight[FIRST][PARTS], first_value[(EP + 255) / 256];
  const uint32_t first_queries = min(16u, per);
  if (RAW) {
#pragma unroll
    for (int j = 0; j < FIRST; ++j) {
      const uint32_t n = min((uint32_t)wave + 4 * j, first_queries);  // (the last one is the key)
      const bool query = n < first_queries;
      const float *source = a.row + (query ? (size_t)(group * per + n) * dim : (size_t)(a.heads + group) * dim);
#pragma unroll
      for (int i = 0; i < PARTS; ++i) first[j].v[i] = lane + 64 * i < dim ? source[lane + 64 * i] : 0.0f;
      HeadVector<PARTS>::norm_weights(query ? a.rotation.q_norm : a.rotation.k_norm, dim, lane, first_weight[j]);
    }
    const float *value = a.row + (size_t)(a.heads + a.kv_heads) * dim + (size_t)group * vdim;
#pragma unroll
    for (int i = 0; i < (EP + 255) / 256; ++i) first_value[i] = tid + 256 * i < vdim ? value[tid + 256 * i] : 0.0f;
  }
  Frag<T> fk[2][ND], reg_v[NE];
#pragma unroll
  for (int kt = 0; kt < 2; ++kt) {
    const T *row = cache_k + (size_t)(min(wave_begin + kt * 16 + column, position) % a.cache.capacity) * dim;
#pragma unroll
    for (int d = 0; d < ND; ++d) fk[kt][d] = load_piece(row + d * 32 + quad * 8, FULL ? 8 : (int)dim - (d * 32 + quad * 8), vec);
  }
#pragma unroll
  for (int i = 0; i < NE; ++i) {
    const int index = i * 64 + lane, row = index / V_PIECES, piece = (index % V_PIECES) * 8;
    const uint32_t j = min(wave_begin + row, position) % a.cache.capacity;
    reg_v[i] = load_piece(cache_v + (size_t)j * vdim + piece, FULL ? 8 : (int)vdim - piece, vec);
  }
  const bool capped = a.softcap > 0.0f;
  const float cap = a.softcap * kLog2e;
  const float inner = capped ? 2.0f * a.scale / a.softcap * kLog2e : a.scale * kLog2e;

  // a raw row: the first sixteen queries and the own key and value
  constexpr int SQ = ND * 32 + 16 / (int)sizeof(T);
  T *lds_q = reinterpret_cast<T *>(lds + decode_lds_floats<T, NE>() * 4), *own_k = lds_q + 16 * SQ, *own_v = own_k + SQ;
  float *exchange = reinterpret_cast<float *>(own_v + EP) + wave * PARTS * 64;
  Turn *turns = reinterpret_cast<Turn *>(reinterpret_cast<float *>(own_v + EP) + 4 * PARTS * 64);
  const ThroughLds<PARTS> partners{exchange, a.rotation.dims, lane};
  auto stage_vector = [&](const HeadVector<PARTS> &h, T *target) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < PARTS; ++i)
      if (lane + 64 * i < ND * 32) target[lane + 64 * i] = (T)h.v[i];  // (zeros behind the head's end)
  };
  // the vectors from `from` on of the queries h0 .. and the key behind them
  auto stage_vectors = [&](uint32_t from, uint32_t h0, uint32_t count, bool key) {
    for (uint32_t n = from + wave; n < count + (key ? 1 : 0); n += 4) {
      const bool query = n < count;
      const float *source = a.row + (query ? (size_t)(group * per + h0 + n) * dim : (size_t)(a.heads + group) * dim);
      HeadVector<PARTS> h;
#pragma unroll
      for (int i = 0; i < PARTS; ++i) h.v[i] = lane + 64 * i < dim ? source[lane + 64 * i] : 0.0f;
      h.norm_and_rotate(a.rotation, query ? a.rotation.q_norm : a.rotation.k_norm, dim, turns, lane, partners);
      stage_vector(h, query ? lds_q + n * SQ : own_k);
    }
  };
  if (RAW) {
    fill_turns(a.rotation, position, turns);
#pragma unroll
    for (int j = 0; j < FIRST; ++j) first[j].normalise(a.rotation, first_weight[j], dim);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < FIRST; ++j) {
      const uint32_t n = wave + 4 * j;
      if (n > first_queries) break;
      first[j].rotate(a.rotation, turns, lane, partners);
      stage_vector(first[j], n < first_queries ? lds_q + n * SQ : own_k);
    }
    stage_vectors(4 * FIRST, 0, first_queries, true);
#pragma unroll
    for (int i = 0; i < (EP + 255) / 256; ++i)
      if (tid + 256 * i < EP) own_v[tid + 256 * i] = (T)first_value[i];  // (zeros behind the value's end)
    __syncthreads();
    if (begin + kSplitKeys > position) {  // this workgroup's keys end with the own one
      const size_t at = ring + position % a.cache.capacity;
      for (uint32_t c = tid; c < dim; c += 256) static_cast<T *>(a.cache.keys)[at * dim + c] = own_k[c];
      for (uint32_t c = tid; c < vdim; c += 256) static_cast<T *>(a.cache.values)[at * vdim + c] = own_v[c];
    }
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
      if (wave_begin + kt * 16 + column >= position)
#pragma unroll
        for (int d = 0; d < ND; ++d) fk[kt][d] = *reinterpret_cast<const Frag<T> *>(own_k + d * 32 + quad * 8);
#pragma unroll
    for (int i = 0; i < NE; ++i) {
      const int index = i * 64 + lane;
      if (wave_begin + index / V_PIECES >= position)
        reg_v[i] = *reinterpret_cast<const Frag<T> *>(own_v + (index % V_PIECES) * 8);
    }
  }

  for (uint32_t h0 = 0; h0 < per; h0 += 16) {
    const uint32_t head = group * per + min(h0 + column, per - 1);
    Frag<T> fq[ND];
    if (RAW && h0 > 0) {
      stage_vectors(0, h0, min(16u, per - h0), false);
      __syncthreads();
    }
#pragma unroll
    for (int d = 0; d < ND; ++d)
      fq[d] = RAW ? *reinterpret_cast<const Frag<T> *>(lds_q + min((uint32_t)column, per - 1 - h0) * SQ + d * 32 + quad * 8)
                  : load_piece(static_cast<const T *>(a.qkv) + (size_t)head * dim + d * 32 + quad * 8,
                               FULL ? 8 : (int)dim - (d * 32 + quad * 8), vec);
    f32x4 score[2];
    float best = -1e30f;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      score[kt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int d = 0; d < ND; ++d) score[kt] = mma(fk[kt][d], fq[d], score[kt]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float s = score[kt][r] * inner;
        if (capped) s = fmaf(-2.0f * cap, __builtin_amdgcn_rcpf(1.0f + exp2_raw(s)), cap);
        if (wave_begin + kt * 16 + quad * 4 + r > position) s = -INFINITY;
        score[kt][r] = s;
        best = fmaxf(best, s);
      }
    }
    best = fmaxf(best, __shfl_xor(best, 16, 64));
    best = fmaxf(best, __shfl_xor(best, 32, 64));
    if (quad == 0) lds_top[wave * 16 + column] = best;
#pragma unroll
    for (int i = 0; i < NE; ++i) {
      const int index = i * 64 + lane;
      *reinterpret_cast<Frag<T> *>(lds_v + index / V_PIECES * SV + (index % V_PIECES) * 8) = reg_v[i];
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 4; ++w) best = fmaxf(best, lds_top[w * 16 + column]);
    WideFrag<T> fp;
    float total = 0.0f;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float p = exp2_raw(score[kt][r] - best);
        total += p;
        fp.set(kt * 4 + r, p);
      }
    total += __shfl_xor(total, 16, 64);
    total += __shfl_xor(total, 32, 64);
    if (quad == 0) lds_total[wave * 16 + column] = total;
    f32x4 out[NE];
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      const T *keys = lds_v + quad * 4 * SV + e * 16;
      const auto first = four_keys(keys, SV, lane), second = four_keys(keys + 16 * SV, SV, lane);
      const Frag<T> fv = __builtin_shufflevector(first, second, 0, 1, 2, 3, 4, 5, 6, 7);
      out[e] = mma_wide_b(fv, fp, f32x4{0.0f, 0.0f, 0.0f, 0.0f});
    }
    __syncthreads();  // every read of the values is done
#pragma unroll
    for (int e = 0; e < NE; ++e)
      *reinterpret_cast<f32x4 *>(lds + wave * OWN + (column * EP + e * 16 + quad * 4) * 4) = out[e];
    __syncthreads();
    const uint32_t live = min(16u, per - h0);
    for (uint32_t i = tid; i < live * EP; i += 256) {
      const uint32_t h = i / EP, c = i % EP;
      if (c >= vdim) continue;
      float sum = 0.0f, all = 0.0f, top = -1e30f;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        sum += *reinterpret_cast<const float *>(lds + w * OWN + (h * EP + c) * 4);
        all += lds_total[w * 16 + h];
        top = fmaxf(top, lds_top[w * 16 + h]);
      }
      const uint32_t target = group * per + h0 + h;
      if (alone) {
        if (a.sink) {
          const float sink = (float)reinterpret_cast<const __bf16 *>(a.sink)[target] * kLog2e, most = fmaxf(top, sink);
          const float mine = exp2_raw(top - most);
          sum *= mine;
          all = fmaf(all, mine, exp2_raw(sink - most));
        }
        store_attention<T>(a, target, c, sum / all);
      } else {
        float *partial = static_cast<float *>(a.workspace) + ((size_t)target * splits + split) * (vdim + 2);
        const auto leave = [](float *to, float v) {
          if (JOIN) hand_over(to, v);
          else *to = v;
        };
        leave(partial + c, sum);
        if (c == 0) {
          leave(partial + vdim, top);
          leave(partial + vdim + 1, all);
        }
      }
    }
    __syncthreads();
  }
  if (JOIN && !alone) join_shares<T>(a, splits, group, live, counters + group, lds);
}

// 256 threads a head; the splits' weights are formed once, in LDS (two words a split; maxima are exponents of two).
template <typename T>
__device__ __forceinline__ void chunk_merge(const ChunkAttentionArgs &a, uint32_t splits, uint32_t head, float *shared) {
  float *best = shared, *total = shared + splits;
  const uint32_t position = a.state[kStatePosition];
  const uint32_t live = min(splits, (position - first_seen(position, a.cache)) / kSplitKeys + 1);
  const uint32_t stride = a.vdim + 2;
  const float *partial = static_cast<const float *>(a.workspace) + (size_t)head * splits * stride;
  const float sink = a.sink ? (float)reinterpret_cast<const __bf16 *>(a.sink)[head] * kLog2e : -INFINITY;
  constexpr uint32_t AHEAD = 8;
  const uint32_t c = threadIdx.x;
  float first[AHEAD];  // the first splits' values on their way while the weights are formed
#pragma unroll
  for (uint32_t s = 0; s < AHEAD; ++s) first[s] = s < live && c < a.vdim ? partial[s * stride + c] : 0.0f;
  for (uint32_t s = threadIdx.x; s < live; s += 256) {
    best[s] = partial[s * stride + a.vdim];
    total[s] = partial[s * stride + a.vdim + 1];
  }
  __syncthreads();
  float top = sink;
  for (uint32_t s = 0; s < live; ++s) top = fmaxf(top, best[s]);
  float denominator = exp2_raw(sink - top), sum = 0.0f;
#pragma unroll
  for (uint32_t s = 0; s < AHEAD; ++s)
    if (s < live) {
      const float weight = exp2_raw(best[s] - top);
      denominator = fmaf(total[s], weight, denominator);
      sum = fmaf(first[s], weight, sum);
    }
#pragma unroll 8
  for (uint32_t s = AHEAD; s < live; ++s) {
    const float weight = exp2_raw(best[s] - top);
    denominator = fmaf(total[s], weight, denominator);
    if (c < a.vdim) sum = fmaf(partial[s * stride + c], weight, sum);
  }
  if (c >= a.vdim) return;
  store_attention<T>(a, head, c, sum / denominator);
}

template <typename T, int ND, int NE>
bool full_heads(const ChunkAttentionArgs &a) {
  return sizeof(T) == 2 && a.dim == ND * 32 && a.vdim == NE * 16;
}

// Most shares of 128 keys that a token can have.
inline uint32_t decode_splits(const ChunkAttentionArgs &a) {
  const uint32_t span = a.cache.span, capacity = a.cache.capacity, longest = span && span < capacity ? span : capacity;
  return (longest + kSplitKeys - 1) / kSplitKeys;
}

inline bool joins_shares(const ChunkAttentionArgs &a) {
  return a.counters != nullptr && joins(decode_splits(a), a.heads, a.kv_heads, a.vdim, a.counter_count, decode_lds_floats<__bf16, 2>());
}

}  // namespace llmopt
