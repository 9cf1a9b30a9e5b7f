// Grouped-query attention over chunks of positions or a sliding window, with a tanh cap on the scores and a
// learned sink in the softmax denominator (both optional).
//
//   score(i, j) = cap tanh(scale q_i . k_j / cap),  visible when j <= i and i / chunk == j / chunk,
//                                                   or when 0 <= i - j < window
//   out_i = sum_j exp(score) v_j / (sum_j exp(score) + exp(sink))
//
// Keys and values live in a ring per sequence slot and head: position p in row p % capacity, capacity >=
// chunk or window, so that a ring of one holds everything later tokens can see.
//
//  * chunk_turns_kernel: a portion of a prompt in bfloat16 whose rows walk over many keys; described at the kernel.
//  * chunk_prefill_kernel: any other portion of a prompt.  Waves of 16 query rows of one head each walk its keys,
//    64 keys a stage through LDS; keys before the portion come from the ring, the others from the
//    portion's own rows.  Bound by the latency of a stage (products, softmax, products in turn): matrix units are
//    busy for 29% of the time and vector units for 50%, and a second stage in LDS gives nothing.  16 heads of 128
//    over 3001 rows take 92 us (138 with four waves of 32 rows): 119 with eight waves of 16 rows a workgroup, four a
//    SIMD, 112 with tiles dealt as below, 96 with the border mask behind its own branch, 92 with the weights' parts
//    converted in pairs.  S^T = K Q^T leaves every lane four consecutive keys of one query row, which is
//    the B operand of O^T += V^T P^T up to a permutation of the contraction index that the V^T operand
//    follows: probabilities never leave their lane (bf16: as a high and a low part, so that the weights keep
//    float32 accuracy in the product).  Caps of at most kFixedMaxCap bound the exponent, so
//    the running maximum (and the rescaling) is dropped for a constant one.
//  * chunk_decode_kernel: one token.  A workgroup takes kSplitKeys keys of one key / value head for all
//    query heads on it, which are the operand columns; where the ring is longer than one split the last workgroup of a
//    head joins them, or chunk_merge_kernel (joins_shares:
//    the line between them).  Over a raw float32 row it norms and rotates the group's queries and the token's own
//    key first (in LDS) and leaves key and value in the ring; the own key and value never come from there.
//  * rotate_heads_kernel: the same norm and rotation for a portion of a prompt, in place.
#include <algorithm>
#include <cfloat>
#include <type_traits>

#include "attention_turns.h"
#include "chunk_decode.h"
#include "dense_attention_rule.h"
#include "dense.h"
#include "dense_common.h"
#include "kernels_internal.h"

namespace llmopt {

template <>
struct TurnsOperand<__bf16> {
  typedef bf16x8 x8;
  typedef WideFrag<__bf16> Weights;  // the weights keep float32 accuracy
  static constexpr int kProducts = 2;
  static __device__ __forceinline__ f32x16 product(x8 a, x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x16 weighted(x8 a, const Weights &w, f32x16 c) {
    return product(a, w.lo, product(a, w.hi, c));
  }
};

namespace {

constexpr int kStageKeys = 64;
constexpr float kFixedMaxCap = 40.0f;

// The stage, and where KS == 2 the second half's sums in its place.
template <typename T, int ND, int NE, int WAVES, int KS>
constexpr int prefill_lds_bytes() {
  const int stage = kStageKeys * (ND * 32 + 16 / (int)sizeof(T) + value_stride<T, NE>()) * (int)sizeof(T);
  const int sums = KS == 2 ? WAVES / 2 * 64 * (NE * 4 + 2) * 4 : 0;
  return stage > sums ? stage : sums;
}

// Eight waves keep to the registers that let a compute unit hold two workgroups.
template <typename T, int ND, int NE, int WAVES, int KS, bool FIXED>
__global__ __launch_bounds__(WAVES * 64, WAVES == 8 ? 4 : ND * 2 + NE <= 16 || sizeof(T) == 2 ? 2 : 1) void
chunk_prefill_kernel(ChunkAttentionArgs a, uint32_t cus) {
  constexpr int DP = ND * 32, EP = NE * 16;
  constexpr int ROW_WAVES = WAVES / KS, ROWS = ROW_WAVES * 16, KEYS = kStageKeys / KS, KT = KEYS / 16;
  constexpr int SK = DP + 16 / (int)sizeof(T), SV = value_stride<T, NE>();
  constexpr int K_LOADS = kStageKeys * DP / 8 / (WAVES * 64), V_PIECES = EP / 8;
  constexpr int V_LOADS = (kStageKeys * V_PIECES + WAVES * 64 - 1) / (WAVES * 64);
  extern __shared__ __attribute__((aligned(16))) char lds[];
  T *lds_k = reinterpret_cast<T *>(lds);
  T *lds_v = lds_k + kStageKeys * SK;

  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int column = lane & 15, quad = lane >> 4, row_wave = wave % ROW_WAVES, first_key = wave / ROW_WAVES * KEYS;
  // Heads of one key / value head follow each other kv_heads apart, so that they share an XCD's L2 when
  // kv_heads is a multiple of the eight XCDs.  Late rows see more keys: tiles are dealt in rounds of one
  // workgroup a compute unit, the longest round first, and in turn from short to long and from long to short, so
  // that the second workgroup of a compute unit is short where its first one is long (16 heads of 3001 rows: 119 us
  // with the longest first, 112 so).
  const uint32_t per = a.heads / a.kv_heads, group = blockIdx.x % a.kv_heads;
  const uint32_t head = group * per + blockIdx.x / a.kv_heads;
  const uint32_t around = max(cus / a.heads, 1u), round = blockIdx.y / around, step = blockIdx.y % around;
  const uint32_t left = gridDim.y - round * around;  // tiles of this round and later ones
  const uint32_t p0 = a.state[kStatePosition], slot = a.state[kStateSlot];
  uint32_t tile = gridDim.y <= around || (round & 1) ? left - 1 - step : left - min(left, around) + step;
  if constexpr (sizeof(T) == 4) {
    if (gridDim.y > around && gridDim.y <= 64 && !a.cache.sliding && a.cache.span != 0 &&
        first_seen(p0, a.cache) + a.cache.span < p0 + a.m) {
      // A chunk ends inside the portion, and the rows behind it start from nothing: the same rounds over the tiles in the
      // order of their keys (1024 rows of 32 heads of 128 from position 1500 on, chunks of 2048: 332 us as if late rows saw
      // more, 296 with the last rows first, 269 so; 300 rows of 64 heads, chunks of 512: 98, 84, 71).  Lane t ranks tile t.
      // (With no such chunk the wait for the position costs what 1024 rows of 64 heads show most, 205 us without, 216 with;
      // bfloat16's stages are too short for it.)
      const uint32_t first = p0 + min(lane * ROWS, (int)a.m - 1), keys = min(first + ROWS, p0 + a.m) - first_seen(first, a.cache);
      uint32_t longer = 0;
      for (uint32_t t = 0; t < gridDim.y; ++t) {
        const uint32_t its = __builtin_amdgcn_readlane(keys, t);
        longer += its > keys || (its == keys && (int)t > lane);
      }
      tile = __builtin_ctzll(__ballot(longer == gridDim.y - 1 - tile && lane < (int)gridDim.y));
    }
  }
  const uint32_t row_first = tile * ROWS;
  const uint32_t row_end = min(row_first + ROWS, a.m);
  const uint32_t ld = a.ld;
  const T *qkv = static_cast<const T *>(a.qkv);
  const T *fresh_k = qkv + a.heads * a.dim + group * a.dim;
  const T *fresh_v = qkv + a.heads * a.dim + a.kv_heads * a.dim + group * a.vdim;
  const size_t ring = ((size_t)slot * a.kv_heads + group) * a.cache.capacity;
  const T *cache_k = static_cast<const T *>(a.cache.keys) + ring * a.dim;
  const T *cache_v = static_cast<const T *>(a.cache.values) + ring * a.vdim;
  const bool vec = a.dim % 8 == 0 && a.vdim % 8 == 0 && ld % 8 == 0;

  // queries of this wave: operand columns
  Frag<T> fq[ND];
  const uint32_t row = row_first + row_wave * 16 + column, own = min(row, a.m - 1);
  const uint32_t query = p0 + own, low = first_seen(query, a.cache);  // visible positions of the lane's row: low .. query
#pragma unroll
  for (int d = 0; d < ND; ++d) {
    const int k = d * 32 + quad * 8;
    fq[d] = load_piece(qkv + (size_t)own * ld + head * a.dim + k, (int)a.dim - k, vec);
  }
  const uint32_t wave_first = p0 + min(row_first + row_wave * 16, a.m - 1);
  const uint32_t wave_last = p0 + min(row_first + (row_wave + 1) * 16 - 1, a.m - 1);
  const uint32_t wave_low = first_seen(wave_first, a.cache);
  const uint32_t wave_low_last = first_seen(wave_last, a.cache);

  // Exponents are taken to base two.  capped: score = cap tanh(scale s / cap), with
  // tanh z = 1 - 2 / (1 + e^(2 z)); fixed: the cap bounds it, and the maximum is a constant.
  const bool has_sink = a.sink != nullptr, capped = a.softcap > 0.0f;
  const float sink = has_sink ? (float)reinterpret_cast<const __bf16 *>(a.sink)[head] * kLog2e : 0.0f;
  const float cap = a.softcap * kLog2e;
  const float inner = capped ? 2.0f * a.scale / a.softcap * kLog2e : a.scale * kLog2e;
  float top = FIXED ? fmaxf(sink, 0.0f) : first_key == 0 && has_sink ? sink : -1e30f;
  float total = has_sink && first_key == 0 && quad == 0 ? exp2_raw(sink - top) : 0.0f;
  f32x4 out[NE];
#pragma unroll
  for (int e = 0; e < NE; ++e) out[e] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  const uint32_t last = p0 + row_end - 1;
  const uint32_t key_begin = first_seen(p0 + row_first, a.cache);

  // a stage travels global -> registers while the one before it is multiplied
  Frag<T> reg_k[K_LOADS], reg_v[V_LOADS];
  auto fetch = [&](uint32_t base) {
#pragma unroll
    for (int i = 0; i < K_LOADS; ++i) {
      const int index = i * WAVES * 64 + tid, row = index / (DP / 8), piece = (index % (DP / 8)) * 8;
      const uint32_t j = min(base + row, last);
      const T *source = j < p0 ? cache_k + (size_t)(j % a.cache.capacity) * a.dim : fresh_k + (size_t)(j - p0) * ld;
      reg_k[i] = load_piece(source + piece, (int)a.dim - piece, vec);
    }
#pragma unroll
    for (int i = 0; i < V_LOADS; ++i) {
      const int index = i * WAVES * 64 + tid, row = min(index / V_PIECES, kStageKeys - 1), piece = (index % V_PIECES) * 8;
      const uint32_t j = min(base + row, last);
      const T *source = j < p0 ? cache_v + (size_t)(j % a.cache.capacity) * a.vdim : fresh_v + (size_t)(j - p0) * ld;
      reg_v[i] = load_piece(source + piece, (int)a.vdim - piece, vec);
    }
  };
  auto stash = [&] {
#pragma unroll
    for (int i = 0; i < K_LOADS; ++i) {
      const int index = i * WAVES * 64 + tid;
      *reinterpret_cast<Frag<T> *>(lds_k + index / (DP / 8) * SK + (index % (DP / 8)) * 8) = reg_k[i];
    }
#pragma unroll
    for (int i = 0; i < V_LOADS; ++i) {
      const int index = i * WAVES * 64 + tid;
      if (index < kStageKeys * V_PIECES)
        *reinterpret_cast<Frag<T> *>(lds_v + index / V_PIECES * SV + (index % V_PIECES) * 8) = reg_v[i];
    }
  };

  auto multiply = [&](uint32_t base) {  // base: the first of this wave's keys in the stage
    f32x4 score[KT];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) score[kt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int d = 0; d < ND; ++d) {
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) {
        const Frag<T> fk = *reinterpret_cast<const Frag<T> *>(lds_k + (first_key + kt * 16 + column) * SK + d * 32 + quad * 8);
        score[kt] = mma(fk, fq[d], score[kt]);
      }
      if (KS == 1) __builtin_amdgcn_sched_barrier(0);  // four operands at a time: registers
    }
    // Only a stage with a border pays for the mask: behind its own branch, which all of a wave takes alike (with a
    // test beside each score 16 heads of 3001 rows took 114 us for 96).
    const bool whole = base >= wave_low_last && base + KEYS - 1 <= wave_first;
    auto mask = [&](float hidden) {
      const uint32_t from = low - base - quad * 4, count = query - low;
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) score[kt][r] = kt * 16 + r - from <= count ? score[kt][r] : hidden;
    };
    if (FIXED) {
      const float high = cap - top;
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float tail = __builtin_amdgcn_rcpf(1.0f + exp2_raw(score[kt][r] * inner));
          score[kt][r] = exp2_raw(fmaf(-2.0f * cap, tail, high));
        }
      if (!whole) mask(0.0f);
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) total += score[kt][r];
    } else {
      if (capped) {
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            score[kt][r] = fmaf(-2.0f * cap, __builtin_amdgcn_rcpf(1.0f + exp2_raw(score[kt][r] * inner)), cap);
      } else {
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) score[kt] *= inner;
      }
      if (!whole) mask(-INFINITY);
      float best = top;
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) best = fmaxf(best, score[kt][r]);
      best = fmaxf(best, __shfl_xor(best, 16, 64));
      best = fmaxf(best, __shfl_xor(best, 32, 64));
      const float alpha = exp2_raw(top - best);
      top = best;
      total *= alpha;
#pragma unroll
      for (int e = 0; e < NE; ++e) out[e] *= alpha;
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          score[kt][r] = exp2_raw(score[kt][r] - best);
          total += score[kt][r];
        }
    }
#pragma unroll
    for (int ks = 0; ks < KT / 2; ++ks) {
      WideFrag<T> fp;  // the weights keep float32 accuracy
#pragma unroll
      for (int r = 0; r < 4; r += 2) {
        fp.set_pair(r, score[2 * ks][r], score[2 * ks][r + 1]);
        fp.set_pair(4 + r, score[2 * ks + 1][r], score[2 * ks + 1][r + 1]);
      }
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        const T *keys = lds_v + (first_key + ks * 32 + quad * 4) * SV + e * 16;
        const auto first = four_keys(keys, SV, lane), second = four_keys(keys + 16 * SV, SV, lane);
        const Frag<T> fv = __builtin_shufflevector(first, second, 0, 1, 2, 3, 4, 5, 6, 7);
        out[e] = mma_wide_b(fv, fp, out[e]);
        if (e % 4 == 3) __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  fetch(key_begin);
  for (uint32_t base = key_begin; base <= last; base += kStageKeys) {
    __syncthreads();
    stash();
    __syncthreads();
    if (base + kStageKeys <= last) fetch(base + kStageKeys);
    const uint32_t begin = base + first_key;
    if (begin <= wave_last && begin + KEYS > wave_low) multiply(begin);
  }

  if constexpr (KS == 2) {  // the second half's sums join the first's through the stage's LDS
    constexpr int WORDS = NE * 4 + 2;
    float *other = reinterpret_cast<float *>(lds) + row_wave * 64 * WORDS + lane;
    __syncthreads();
    if (first_key) {
#pragma unroll
      for (int e = 0; e < NE; ++e)
#pragma unroll
        for (int r = 0; r < 4; ++r) other[(e * 4 + r) * 64] = out[e][r];
      other[NE * 4 * 64] = top;
      other[(NE * 4 + 1) * 64] = total;
    }
    __syncthreads();
    if (first_key) return;
    const float its_top = other[NE * 4 * 64], best = fmaxf(top, its_top);
    const float mine = exp2_raw(top - best), its = exp2_raw(its_top - best);
    total = total * mine + other[(NE * 4 + 1) * 64] * its;
#pragma unroll
    for (int e = 0; e < NE; ++e)
#pragma unroll
      for (int r = 0; r < 4; ++r) out[e][r] = out[e][r] * mine + other[(e * 4 + r) * 64] * its;
  }
  float sum = total;
  sum += __shfl_xor(sum, 16, 64);
  sum += __shfl_xor(sum, 32, 64);
  const float inverse = a.out_scale / sum;
  if (row >= a.m) return;
  T *target = static_cast<T *>(a.out) + (size_t)row * a.ld_out + head * a.vdim;
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    const uint32_t c = e * 16 + quad * 4;
    typedef T x4 __attribute__((ext_vector_type(4)));
    if (vec && a.ld_out % 4 == 0 && c < a.vdim) {
      x4 packed;
#pragma unroll
      for (int i = 0; i < 4; ++i) packed[i] = (T)(out[e][i] * inverse);
      *reinterpret_cast<x4 *>(target + c) = packed;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (c + i < a.vdim) target[c + i] = (T)(out[e][i] * inverse);
    }
  }
}

// A long portion of a prompt, bfloat16: 32 rows a wave and two groups of waves in turns (attention_turns.h), the keys of 128 rows
// shared between them.  Bound by both sides of a turn alike: 48 products of 64 keys, of which the weights' low part is a third,
// take 2050 cycles beside the other wave's softmax and split (1500 and 250 of copies; under a cap 2650), 1536 by themselves.
// 16 heads of 128 over 3001 rows with a window of 2048, norm and cache writes included: 96 -> 75 us; 32 heads over 2048 under a
// cap 90 -> 74.  The weights packed beside the products instead: 77 / 81 for 74 / 76.
template <int D, TurnsScores SCORES>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void chunk_turns_kernel(ChunkAttentionArgs a) {
  constexpr int JJ = D / 32, WAVES = 4;
  constexpr uint32_t ROWS = turns_rows<true>();
  extern __shared__ __attribute__((aligned(16))) unsigned char stage_lds[];
  const uint32_t lane = threadIdx.x & 63, row_lane = lane & 31, half = lane >> 5;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t slabs = (a.m + ROWS - 1) / ROWS, within = blockIdx.x % a.heads, slab = slabs - 1 - blockIdx.x / a.heads;
  const uint32_t per = a.heads / a.kv_heads, kv_head = within % a.kv_heads, head = kv_head * per + within / a.kv_heads;
  const uint32_t p0 = a.state[kStatePosition], slot = a.state[kStateSlot], ld = a.ld, capacity = a.cache.capacity;
  const uint32_t wave_row = slab * ROWS + wave % WAVES * 32, own = min(wave_row + row_lane, a.m - 1);
  const __bf16 *qkv = static_cast<const __bf16 *>(a.qkv);

  bf16x8 q[D / 16];
  const __bf16 *q_row = qkv + (size_t)own * ld + head * D;
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks) q[ks] = *reinterpret_cast<const bf16x8 *>(q_row + ks * 16 + half * 8);
  const uint32_t first_row = p0 + min(wave_row, a.m - 1), last_row = p0 + min(wave_row + 31, a.m - 1);
  const TurnsBounds bounds = {first_seen(p0 + own, a.cache), p0 + own, first_seen(first_row, a.cache), first_seen(last_row, a.cache),
                              first_row, last_row, wave_row < a.m};
  const uint32_t last = p0 + min(slab * ROWS + ROWS, a.m) - 1, begin = first_seen(p0 + slab * ROWS, a.cache);

  const __bf16 *fresh_k = qkv + (a.heads + kv_head) * D, *fresh_v = fresh_k + a.kv_heads * D;
  const size_t ring = ((size_t)slot * a.kv_heads + kv_head) * capacity * D;
  const __bf16 *cache_k = static_cast<const __bf16 *>(a.cache.keys) + ring, *cache_v = static_cast<const __bf16 *>(a.cache.values) + ring;
  const TurnsCopy<D, WAVES, false> k_rows(ld * 2, threadIdx.x);
  const TurnsCopy<D, WAVES, true> v_rows(ld * 2, threadIdx.x);
  // a row of a stage that begins before the portion or goes beyond its last row, which is then repeated
  const auto row_of = [&](const __bf16 *fresh, const __bf16 *cache, uint32_t key, uint32_t r) {
    const uint32_t j = min(key + r, last);
    uint32_t at = key % capacity + (j - key);
    at -= at >= capacity ? capacity : 0;
    return j < p0 ? cache + (size_t)at * D : fresh + (size_t)(j - p0) * ld;
  };
  const auto copy = [&](const auto &rows, const __bf16 *fresh, const __bf16 *cache, uint32_t key, uint32_t stage) {
    const uint32_t at = key % capacity;
    if (key >= p0 && key + kTurnsKeys - 1 <= last) {
      rows.whole(fresh + (size_t)(key - p0) * ld, stage);
    } else if (key + kTurnsKeys <= p0 && at + kTurnsKeys <= capacity) {
      uint32_t thread = threadIdx.x;
      asm volatile("" : "+v"(thread));  // (made anew: these stages are the earlier portions' only)
      std::decay_t<decltype(rows)>(D * 2, thread).whole(cache + (size_t)at * D, stage);
    } else {
      rows.rows([&](uint32_t r) { return row_of(fresh, cache, key, r); }, stage);
    }
  };
  const auto copy_k = [&](uint32_t key, uint32_t stage) { copy(k_rows, fresh_k, cache_k, key, stage); };
  const auto copy_v = [&](uint32_t key, uint32_t stage) { copy(v_rows, fresh_v, cache_v, key, stage); };

  const bool has_sink = a.sink != nullptr && wave < WAVES;
  const float sink = has_sink ? (float)reinterpret_cast<const __bf16 *>(a.sink)[head] * kLog2e : -FLT_MAX;
  const float inner = (SCORES == TurnsScores::kPlain ? a.scale : 2.0f * a.scale / a.softcap) * kLog2e;
  float top = SCORES == TurnsScores::kFixed ? fmaxf(sink, 0.0f) : sink;
  float total = has_sink && half == 0 ? exp2_raw(sink - top) : 0.0f;
  f32x16 out[JJ];
#pragma unroll
  for (int jj = 0; jj < JJ; ++jj)
#pragma unroll
    for (int r = 0; r < 16; ++r) out[jj][r] = 0.0f;
  if (!attention_turns<__bf16, D, true, SCORES>(stage_lds, q, bounds, begin, (last - begin) / kTurnsKeys + 1, inner,
                                                 a.softcap * kLog2e, top, total, out, copy_k, copy_v))
    return;
  float low, high;
  both_halves(total, low, high);
  const float inverse = a.out_scale / (low + high);
  if (wave_row >= a.m) return;
  constexpr int FROM = turns_share_bytes<D>();
  static_assert(FROM + WAVES * store_rows_bytes<D>() <= turns_lds_bytes<D, true>(), "the rows fit the stages");
  store_rows<D>(stage_lds + FROM + wave * store_rows_bytes<D>(), static_cast<__bf16 *>(a.out) + (size_t)wave_row * a.ld_out + head * D,
                (size_t)a.ld_out * 2, a.m - wave_row, [&](int jj, int r) {
                  bf16x4 packed;
#pragma unroll
                  for (int i = 0; i < 4; ++i) packed[i] = (__bf16)(out[jj][r + i] * inverse);
                  return __builtin_bit_cast(uint2, packed);
                });
}

template <typename T>
__global__ __launch_bounds__(256) void chunk_cache_write_kernel(ChunkAttentionArgs a, uint32_t first_row) {
  const uint32_t r = first_row + blockIdx.x;
  const uint32_t position = a.state[kStatePosition] + r, slot = a.state[kStateSlot];
  const uint32_t row = position % a.cache.capacity;
  const uint32_t n_k = a.kv_heads * a.dim, n_v = a.kv_heads * a.vdim;
  const T *source = static_cast<const T *>(a.qkv) + (size_t)r * a.ld + a.heads * a.dim;
  T *keys = static_cast<T *>(a.cache.keys), *values = static_cast<T *>(a.cache.values);
  for (uint32_t c = threadIdx.x; c < n_k + n_v; c += 256) {
    if (c < n_k)
      keys[(((size_t)slot * a.kv_heads + c / a.dim) * a.cache.capacity + row) * a.dim + c % a.dim] = source[c];
    else
      values[(((size_t)slot * a.kv_heads + (c - n_k) / a.vdim) * a.cache.capacity + row) * a.vdim + (c - n_k) % a.vdim] =
          source[c];
  }
}

// A workgroup a row; its waves take vectors 0 .. heads + kv_heads - 1 (the queries, then the keys) in turn, the next one
// requested ahead.
template <typename T, int PARTS>
__global__ __launch_bounds__(256) void rotate_heads_kernel(ChunkAttentionArgs a) {
  __shared__ float rows[4][PARTS * 64];
  __shared__ Turn turns[PARTS * 32];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const uint32_t r = blockIdx.x, vectors = a.heads + a.kv_heads;
  T *row = const_cast<T *>(static_cast<const T *>(a.qkv)) + (size_t)r * a.ld;
  T ahead[PARTS];
  auto request = [&](uint32_t vector) {
#pragma unroll
    for (int i = 0; i < PARTS; ++i)
      if (lane + 64 * i < a.dim) ahead[i] = row[(size_t)vector * a.dim + lane + 64 * i];
  };
  request(min((uint32_t)wave, vectors - 1));
  fill_turns(a.rotation, a.state[kStatePosition] + r, turns);
  __syncthreads();
  for (uint32_t vector = wave; vector < vectors; vector += 4) {
    HeadVector<PARTS> h;
#pragma unroll
    for (int i = 0; i < PARTS; ++i) h.v[i] = lane + 64 * i < a.dim ? to_f32(ahead[i]) : 0.0f;
    request(min(vector + 4, vectors - 1));
    h.norm_and_rotate(a.rotation, vector < a.heads ? a.rotation.q_norm : a.rotation.k_norm, a.dim, turns, lane,
                      ThroughLds<PARTS>{rows[wave], a.rotation.dims, lane});
#pragma unroll
    for (int i = 0; i < PARTS; ++i)
      if (lane + 64 * i < a.dim) row[(size_t)vector * a.dim + lane + 64 * i] = (T)h.v[i];
  }
}

// The same for bfloat16 heads of 8 LANES values: eight values a lane (16-byte accesses), 64 / LANES vectors a wave at once, and a
// wave a row, so that the workgroup's threads share the turns of four rows.  Partners are whole lanes away.  A workgroup a row
// spent its time on one wave's turns and on five trips through LDS behind them: 3001 rows of 20 vectors of 128 18.1 us / 10.1.
template <int LANES>
__global__ __launch_bounds__(256) void rotate_rows_kernel(ChunkAttentionArgs a) {
  constexpr int DIM = LANES * 8, VECTORS = 64 / LANES;
  __shared__ __attribute__((aligned(16))) Turn turns[4][DIM / 2];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, piece = lane % LANES, own = lane / LANES;
  const uint32_t first = blockIdx.x * 4, r = first + wave, vectors = a.heads + a.kv_heads, half = a.rotation.dims / 2;
  __bf16 *row = const_cast<__bf16 *>(static_cast<const __bf16 *>(a.qkv)) + (size_t)min(r, a.m - 1) * a.ld + piece * 8;
  auto request = [&](uint32_t vector) { return *reinterpret_cast<const bf16x8 *>(row + (size_t)min(vector, vectors - 1) * DIM); };
  bf16x8 ahead = request(own);
  const uint32_t position = a.state[kStatePosition];
  for (uint32_t i = threadIdx.x; i < 4 * half; i += 256)
    turn(position + min(first + i / half, a.m - 1), a.rotation.frequencies[i % half], turns[i / half][i % half].cosine,
         turns[i / half][i % half].sine);
  float gain[2][8];  // of queries and keys
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const bf16x8 g = *reinterpret_cast<const bf16x8 *>((k ? a.rotation.k_norm : a.rotation.q_norm) + piece * 8);
#pragma unroll
    for (int e = 0; e < 8; ++e) gain[k][e] = (float)g[e];
  }
  __syncthreads();
  const uint32_t column = piece * 8;
  const bool turned = column < a.rotation.dims, upper = column >= half;
  const int partner = lane + (turned ? (upper ? -(int)half : (int)half) / 8 : 0);
  float cosine[8], sine[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const Turn t = turned ? turns[wave][column - (upper ? half : 0) + e] : Turn{1.0f, 0.0f};
    cosine[e] = t.cosine;
    sine[e] = upper ? t.sine : -t.sine;
  }
  for (uint32_t base = 0; base < vectors; base += VECTORS) {
    const uint32_t vector = base + own;
    float v[8], sum = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      v[e] = (float)ahead[e];
      sum += v[e] * v[e];
    }
    ahead = request(vector + VECTORS);
#pragma unroll
    for (int lanes = 1; lanes < LANES; lanes *= 2) sum += __shfl_xor(sum, lanes, 64);
    const float inverse = 1.0f / sqrtf(sum / (float)DIM + a.rotation.epsilon);
    bf16x8 out;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] *= inverse * (vector < a.heads ? gain[0][e] : gain[1][e]);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float other = __shfl(v[e], partner, 64);
      out[e] = (__bf16)(v[e] * cosine[e] + other * sine[e]);
    }
    if (vector < vectors && r < a.m) *reinterpret_cast<bf16x8 *>(row + (size_t)vector * DIM) = out;
  }
}

template <typename T, int ND, int NE, bool RAW, bool JOIN, bool FULL>
__global__ __launch_bounds__(256) void chunk_decode_kernel(ChunkAttentionArgs a, uint32_t splits, uint32_t *counters) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  chunk_decode<T, ND, NE, RAW, JOIN, FULL>(a, splits, blockIdx.x, blockIdx.y, lds, counters);
}

template <typename T>
__global__ __launch_bounds__(256) void chunk_merge_kernel(ChunkAttentionArgs a, uint32_t splits) {
  extern __shared__ __attribute__((aligned(16))) float shared[];
  chunk_merge<T>(a, splits, blockIdx.x, shared);
}

template <typename T, int ND, int NE, bool RAW, bool JOIN, bool FULL = false>
hipError_t run_decode(const ChunkAttentionArgs &a, hipStream_t stream) {
  if constexpr (sizeof(T) == 2 && !FULL)
    if (full_heads<T, ND, NE>(a)) return run_decode<T, ND, NE, RAW, JOIN, true>(a, stream);
  static bool allowed[kMaxDevices] = {};
  constexpr int bytes = decode_lds_floats<T, NE>() * 4 + (RAW ? raw_row_lds_bytes<T, ND, NE>() : 0);
  const uint32_t splits = decode_splits(a);
  if (bytes > 64 * 1024)
    if (hipError_t status = allow_dynamic_lds(reinterpret_cast<const void *>(chunk_decode_kernel<T, ND, NE, RAW, JOIN, FULL>), bytes, allowed))
      return status;
  chunk_decode_kernel<T, ND, NE, RAW, JOIN, FULL><<<dim3(a.kv_heads, splits), 256, bytes, stream>>>(a, splits, a.counters);
  if (hipError_t status = hipGetLastError()) return status;
  if (splits > 1 && !JOIN) chunk_merge_kernel<T><<<a.heads, 256, splits * 8, stream>>>(a, splits);
  return hipGetLastError();
}

template <typename T, int ND, int NE, int WAVES, int KS, bool FIXED>
hipError_t run_prefill_kernel(const ChunkAttentionArgs &a, hipStream_t stream) {
  constexpr int bytes = prefill_lds_bytes<T, ND, NE, WAVES, KS>(), rows = WAVES / KS * 16;
  static bool allowed[kMaxDevices] = {};
  const auto kernel = chunk_prefill_kernel<T, ND, NE, WAVES, KS, FIXED>;
  if (bytes > 64 * 1024)
    if (hipError_t status = allow_dynamic_lds(reinterpret_cast<const void *>(kernel), bytes, allowed)) return status;
  kernel<<<dim3(a.heads, (a.m + rows - 1) / rows), WAVES * 64, bytes, stream>>>(a, (uint32_t)device_compute_units());
  return hipGetLastError();
}

template <typename T, int ND, int NE, int WAVES, int KS>
hipError_t run_prefill_tile(const ChunkAttentionArgs &a, hipStream_t stream) {
  if (a.softcap > 0.0f && a.softcap <= kFixedMaxCap) return run_prefill_kernel<T, ND, NE, WAVES, KS, true>(a, stream);
  return run_prefill_kernel<T, ND, NE, WAVES, KS, false>(a, stream);
}

template <int D, TurnsScores SCORES>
hipError_t run_turns_kernel(const ChunkAttentionArgs &a, hipStream_t stream) {
  constexpr int bytes = turns_lds_bytes<D, true>();
  constexpr uint32_t rows = turns_rows<true>();
  static bool allowed[kMaxDevices] = {};
  const auto kernel = chunk_turns_kernel<D, SCORES>;
  if (hipError_t status = allow_dynamic_lds(reinterpret_cast<const void *>(kernel), bytes, allowed)) return status;
  kernel<<<a.heads * ((a.m + rows - 1) / rows), 512, bytes, stream>>>(a);
  return hipGetLastError();
}

template <int D>
hipError_t run_turns(const ChunkAttentionArgs &a, hipStream_t stream) {
  if constexpr (D == 128) {
    if (a.softcap > 0.0f && a.softcap <= kFixedMaxCap) return run_turns_kernel<D, TurnsScores::kFixed>(a, stream);
    if (a.softcap > 0.0f) return run_turns_kernel<D, TurnsScores::kCapped>(a, stream);
  }
  return run_turns_kernel<D, TurnsScores::kPlain>(a, stream);
}

// Whole pieces of sixteen bytes, rows that the ring holds a stage of, and maxima taken before the scale.
bool turns_ok(const ChunkAttentionArgs &a) {
  const auto aligned = [](const void *p, uint32_t bytes) { return (reinterpret_cast<uintptr_t>(p) & (bytes - 1)) == 0; };
  return !a.f32 && a.dim == a.vdim && chunk_turns(a.dim, a.softcap > 0.0f, a.m, a.cache.span, a.heads) &&
         a.cache.capacity >= kTurnsKeys && a.ld % 8 == 0 && a.ld < (1u << 24) && a.ld_out % 4 == 0 && aligned(a.qkv, 16) &&
         aligned(a.cache.keys, 16) && aligned(a.cache.values, 16) && aligned(a.out, 8) &&
         (a.softcap > 0.0f || (a.scale > 0.0f && a.scale < INFINITY));
}

// A wave's registers hold 16 query rows of heads up to 128 twice a SIMD beside a second workgroup (bfloat16); wider
// heads and float32 leave room for four waves.  Eight waves are 128 rows, or 64 rows of which each half of the waves
// takes half the keys of a stage: twice the workgroups, half the chain.  That is the better one while 128-row tiles
// leave compute units with one workgroup or none (700 rows: 16 heads of 128 21.9 us for 28.4, 32 heads 21.9 for
// 30.0; 2048 rows, 16 heads of 64 38.9 for 56.5) and for heads up to 64 always, whose stages are short and whose
// keys are cheap to bring in twice (3001 rows, 16 heads of 64: the same 53 us either way).  Beyond that it brings
// in twice the keys for nothing (3001 rows, 16 heads of 128: 102.7 us for 92.3; 2048 rows, 32 heads: 97.9 for 89.1).
// A grid has at most 65536 rows of workgroups: portions of more 64-row tiles than that take the 128-row ones.
template <typename T, int ND, int NE>
hipError_t run_prefill(const ChunkAttentionArgs &a, hipStream_t stream) {
  if constexpr (sizeof(T) == 2 && ND <= 4 && NE <= 8) {
    const bool many = (uint64_t)a.heads * ((a.m + 127) / 128) > (uint64_t)device_compute_units();
    if ((many && (ND > 2 || NE > 4)) || (a.m + 63) / 64 > 65536) return run_prefill_tile<T, ND, NE, 8, 1>(a, stream);
    return run_prefill_tile<T, ND, NE, 8, 2>(a, stream);
  } else {
    return run_prefill_tile<T, ND, NE, 4, 1>(a, stream);
  }
}

template <typename T, int ND, int NE>
hipError_t run_attention(const ChunkAttentionArgs &a, hipStream_t stream) {
  if constexpr (sizeof(T) == 2 && ((ND == 2 && NE == 4) || (ND == 4 && NE == 8))) {
    if (a.m > 1 && turns_ok(a)) return run_turns<ND * 32>(a, stream);
  }
  if (a.m > 1) return run_prefill<T, ND, NE>(a, stream);
  if (joins_shares(a)) return a.row ? run_decode<T, ND, NE, true, true>(a, stream) : run_decode<T, ND, NE, false, true>(a, stream);
  return a.row ? run_decode<T, ND, NE, true, false>(a, stream) : run_decode<T, ND, NE, false, false>(a, stream);
}

template <typename T, int ND>
hipError_t pick_value_width(const ChunkAttentionArgs &a, hipStream_t stream) {
  if (a.vdim <= 32) return run_attention<T, ND, 2>(a, stream);
  if (a.vdim <= 64) return run_attention<T, ND, 4>(a, stream);
  if (a.vdim <= 128) return run_attention<T, ND, 8>(a, stream);
  return run_attention<T, ND, 16>(a, stream);
}

template <typename T>
hipError_t pick_attention(const ChunkAttentionArgs &a, hipStream_t stream) {
  if (a.dim <= 64) return pick_value_width<T, 2>(a, stream);
  if (a.dim <= 128) return pick_value_width<T, 4>(a, stream);
  return pick_value_width<T, 8>(a, stream);
}

}  // namespace

size_t chunk_attention_workspace_bytes(const ChunkAttentionArgs &a) {
  if (a.m != 1) return 0;
  const uint32_t splits = decode_splits(a);
  return splits > 1 ? (size_t)a.heads * splits * (a.vdim + 2) * 4 : 0;
}

bool chunk_attention_ok(const ChunkAttentionArgs &a) {
  return a.dim <= 256 && a.vdim <= 256 && decode_splits(a) <= 8000;  // (the merge keeps two words a split in LDS)
}

hipError_t launch_chunk_attention(const ChunkAttentionArgs &a, hipStream_t stream) {
  return a.f32 ? pick_attention<float>(a, stream) : pick_attention<__bf16>(a, stream);
}

hipError_t launch_rotate_heads(const ChunkAttentionArgs &a, hipStream_t stream) {
  const dim3 grid(a.m);
  const int parts = a.dim <= 64 ? 1 : a.dim <= 128 ? 2 : 4;
  auto run = [&](auto kernel) {
    kernel<<<grid, 256, 0, stream>>>(a);
    return hipGetLastError();
  };
  const auto aligned = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  if (!a.f32 && (a.dim == 64 || a.dim == 128 || a.dim == 256) && a.rotation.dims % 16 == 0 && a.ld % 8 == 0 && aligned(a.qkv) &&
      aligned(a.rotation.q_norm) && aligned(a.rotation.k_norm)) {
    const auto kernel = a.dim == 64 ? rotate_rows_kernel<8> : a.dim == 128 ? rotate_rows_kernel<16> : rotate_rows_kernel<32>;
    kernel<<<(a.m + 3) / 4, 256, 0, stream>>>(a);
    return hipGetLastError();
  }
  if (a.f32)
    return run(parts == 1 ? rotate_heads_kernel<float, 1> : parts == 2 ? rotate_heads_kernel<float, 2> : rotate_heads_kernel<float, 4>);
  return run(parts == 1 ? rotate_heads_kernel<__bf16, 1> : parts == 2 ? rotate_heads_kernel<__bf16, 2> : rotate_heads_kernel<__bf16, 4>);
}

hipError_t launch_chunk_cache_write(const ChunkAttentionArgs &a, hipStream_t stream) {
  const uint32_t first = a.m > a.cache.capacity ? a.m - a.cache.capacity : 0;
  if (a.f32) chunk_cache_write_kernel<float><<<a.m - first, 256, 0, stream>>>(a, first);
  else chunk_cache_write_kernel<__bf16><<<a.m - first, 256, 0, stream>>>(a, first);
  return hipGetLastError();
}

}  // namespace llmopt
