// All layers of a decode step in one resident launch (gfx950): one new token for each of up to 48 sequences of a W4A16
// transformer with heads of 64 over the grouped-Q8 cache, the arithmetic and the rounding points of the launches that it
// stands for (decode_fused.hip, q8_attention.hip, the W4A16 GEMVs).
//
// What bounds a step of these sizes is not bytes but the chain of dependent launches: at hidden 576 each moves under 1 MB
// and takes 4 to 11 us, of which the boundary, the cold code and the first trips to memory are most.  Here the workgroups
// stay, and what one hands to the others are words of memory that carry their own tag:
//
//   A  norm + QKV + rotation     16 output columns x up to 16 sequences a workgroup
//   B  attention over the cache  one KV head of a run of a sequence's tokens; the new token's K and V into its slot
//   C  merge of the runs         one wave or all eight a (sequence, head)
//   D  output projection + residual, E  norm + gate / up + SwiGLU, F  down projection + residual: as A
//
// A handed-over word is 64 bits, two halves or one float32 and the tag of its layer and step, written and read with
// relaxed device-scope atomics: the reader polls the words that it needs, and a word that carries the tag is there, so a
// hand-over is one store on its way and one load (alone, 16 to 128 workgroups and 256 to 768 words to each: 1.0 to 1.7 us;
// a counter that all workgroups add to takes 0.9 at 16, 1.4 at 64, 2.2 at 128 and 4.0 at 256).  No word is written again before all its readers have read it: to write
// layer l + 1's word a workgroup has seen words that depend, through the phases between, on every reader of layer l's.
//
// Eight waves of a workgroup poll and multiply, eight walk the cache.  A CU's loads return in the order of their requests:
// a polled line that takes 320 cycles takes 810 to 870 beside a stream of other loads from the same CU.  So the polling
// waves request the next use's weights into registers right behind a phase's stores, where they land while the words
// travel (requested once the rows are staged: 388 us instead of 357 for 30 layers of one sequence); the walking waves
// request cache tiles a step ahead, registers to LDS, and help stage the rows of several sequences.
//
// 30 layers, hidden 576, this launch alone: one sequence behind 512 / 2048 / 8192 tokens 348 / 357 / 399 us, 32 sequences
// of 1024 to 2048 tokens 746 us.  Whole steps through a plan, launches / resident: 694 / 394 and 1154 / 803 us.
//
// Waits are bounded: a wave that has polled for `wait_ticks` gives up, sets *failed and polls no more, as does every wave
// that sees the word set; all go on to their end with whatever they hold (numbers only: no address depends on them).  The
// host then runs the step by launches, as it does where a sequence reads a slot that the step itself writes.
#include <algorithm>
#include <type_traits>

#include "kernels.h"
#include "kernels_internal.h"
#include "w4_common.h"

namespace llmopt {
namespace {

constexpr uint32_t kHalf = 512;           // threads that poll and multiply; as many walk the cache
constexpr uint32_t kThreads = 2 * kHalf;
constexpr uint32_t kWaves = 8;            // of either kind
constexpr uint32_t kTile = 16;            // output columns of a product tile, sequences at most
constexpr uint32_t kRowPad = 8;           // halves between activation rows in LDS
constexpr uint32_t kReduceStride = 20;    // floats between a tile's sequences in the waves' sums
constexpr uint32_t kReduceWords = kWaves * kTile * kReduceStride;
constexpr uint32_t kPartWords = 65;       // of a run's head: 64 values and their weight
constexpr uint32_t kSlotCache = 1024;     // slots of a run held in LDS
constexpr uint32_t kLdsMost = 158 * 1024;
constexpr uint32_t kPatchBytes = 2 * 16 * 64 + 64;  // K and V of 16 tokens of a KV head, their scales
constexpr uint32_t kRunStride = 68;       // floats: a wave's 64 values of a head, maximum and sum

// Pointers that have been through memory (the layers' table in LDS) are generic to the compiler, and loads through generic
// pointers count as LDS accesses too: the next wait for LDS would wait for them.
template <typename T>
using Global = const __attribute__((address_space(1))) T *;
template <typename T>
using Local = const __attribute__((address_space(3))) T *;
template <typename T>
__device__ __forceinline__ Global<T> global(const void *pointer) {
  return (Global<T>)reinterpret_cast<uintptr_t>(pointer);
}

// (index: of a word behind a pointer that is the same for the whole wave; in bytes it fits 32 bits, so that the address is
// that pointer in scalar registers and one vector register)
__device__ __forceinline__ uint64_t hand_load(const uint64_t *words, uint32_t index) {
  const uint64_t *word = reinterpret_cast<const uint64_t *>(reinterpret_cast<const uint8_t *>(words) + index * 8);
  return __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void hand_store(uint64_t *words, uint32_t index, uint32_t payload, uint32_t tag) {
  uint64_t *word = reinterpret_cast<uint64_t *>(reinterpret_cast<uint8_t *>(words) + index * 8);
  __hip_atomic_store(word, ((uint64_t)tag << 32) | payload, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A lane's patience.  Each wait is bounded by itself; after one has run out none waits any more.
struct Patience {
  uint32_t *failed;
  uint64_t ticks;
  bool gave_up;
  // Called between polls; true: stop polling.
  __device__ __forceinline__ bool spent(uint32_t polls, uint64_t &since) {
    const uint32_t look = ticks != 0 ? 32 : 0;  // (most waits are over before the clock is looked at; 0: none is waited for)
    if ((polls & 63) != look) return gave_up;
    const uint64_t now = wall_clock64();
    if (polls == look) since = now;
    if (now - since >= ticks || __hip_atomic_load(failed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) {
      __hip_atomic_store(failed, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      gave_up = true;
    }
    return gave_up;
  }
};

// Polls the lane's W words [at[0]] .. [at[W - 1]] until each carries its tag.
template <int W>
__device__ __forceinline__ void await_words(uint64_t (&value)[W], const uint64_t *words, Patience &patience, const uint32_t (&at)[W],
                                            const uint32_t (&tag)[W]) {
  uint64_t since = 0;
  for (uint32_t polls = 0;; ++polls) {
#pragma unroll
    for (int j = 0; j < W; ++j) value[j] = hand_load(words, at[j]);
    uint32_t differ = 0;
#pragma unroll
    for (int j = 0; j < W; ++j) differ |= (uint32_t)(value[j] >> 32) ^ tag[j];
    if (differ == 0 || patience.spent(polls, since)) return;
  }
}
template <int W>
__device__ __forceinline__ void await_words(uint64_t (&value)[W], const uint64_t *words, Patience &patience, const uint32_t (&at)[W],
                                            uint32_t tag) {
  uint32_t tags[W];
#pragma unroll
  for (int j = 0; j < W; ++j) tags[j] = tag;
  await_words(value, words, patience, at, tags);
}

template <int CONTROL>
__device__ __forceinline__ float moved(float value) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, value), CONTROL, 0xF, 0xF, true));
}
// The lane's value and that of the lane 16 (32) away: both, in the same order in either lane.
struct Both {
  float a, b;
};
__device__ __forceinline__ Both across16(float value) {
  const uint32_t bits = __builtin_bit_cast(uint32_t, value);
  const auto two = __builtin_amdgcn_permlane16_swap(bits, bits, false, false);
  return {__builtin_bit_cast(float, (uint32_t)two[0]), __builtin_bit_cast(float, (uint32_t)two[1])};
}
__device__ __forceinline__ Both across32(float value) {
  const uint32_t bits = __builtin_bit_cast(uint32_t, value);
  const auto two = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
  return {__builtin_bit_cast(float, (uint32_t)two[0]), __builtin_bit_cast(float, (uint32_t)two[1])};
}
__device__ __forceinline__ float sum_of_rows(float value) {  // over the four rows of 16 lanes
  const Both near = across16(value);
  const Both far = across32(near.a + near.b);
  return far.a + far.b;
}
__device__ __forceinline__ float max_of_rows(float value) {
  const Both near = across16(value);
  const Both far = across32(fmaxf(near.a, near.b));
  return fmaxf(far.a, far.b);
}
constexpr int kFromNext = 0x101, kFromFourth = 0x104, kFromEighth = 0x128;  // row_shl:1, row_shl:4, row_ror:8

__device__ __forceinline__ uint32_t two_halves(float a, float b) {
  return as_u32(h2_t{(_Float16)a, (_Float16)b});
}

// Words of rows that feed a product hold the columns (c, c + 4) of a run of eight, four words a run: the order in which
// the nibbles of a weight dword decode.  Word w of a row: columns word_column(w) and + 4.
__device__ __forceinline__ uint32_t word_column(uint32_t word) { return (word >> 2) * 8 + (word & 3); }

// How the cached tokens are dealt to the workgroups: every sequence at least one run, more in proportion to its context,
// runs of whole 16-token tiles.  Every wave works it out for itself, a sequence a lane (m <= 48), with the same result.
struct Runs {
  uint32_t first, count, tokens, past, offset;  // of the lane's sequence
};
__device__ __forceinline__ uint32_t wave_inclusive(uint32_t value) {
  int v = (int)value;
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);
  return (uint32_t)v;
}
__device__ __forceinline__ Runs deal_runs(const ResidentArgs &a, uint32_t workgroups, uint32_t least) {
  const uint32_t lane = threadIdx.x & 63;
  Runs r = {0, 0, kTile, 0, 0};
  if (lane < a.m) {
    r.past = min(a.past_lengths[lane], a.max_past);
    r.offset = a.slot_offsets[lane];
  }
  const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)wave_inclusive(r.past), 63);
  // (a hair below, so that the shares add up to the workgroups at most whatever the float roundings do)
  const float ratio = total != 0 ? __fmul_rn(__fdiv_rn((float)(workgroups - a.m), (float)total), 0.999999f) : 0.0f;
  const uint32_t share = 1 + (uint32_t)__fmul_rn((float)r.past, ratio);
  r.tokens = max(least, ((r.past + share - 1) / share + kTile - 1) & ~(kTile - 1));
  r.count = lane < a.m ? max(1u, (r.past + r.tokens - 1) / r.tokens) : 0;
  r.first = wave_inclusive(r.count) - r.count;
  return r;
}

// A workgroup's run of one sequence's tokens.
struct Run {
  uint32_t sequence, length;
  Global<uint32_t> slots;
  Local<uint32_t> slot_cache;
  __device__ __forceinline__ uint32_t slot(uint32_t token) const {
    uint32_t slot = slot_cache[min(token, kSlotCache - 1)];
    if (token >= kSlotCache) slot = slots[token];
    return slot;
  }
};

typedef uint32_t cache_u32x4_t __attribute__((ext_vector_type(4), aligned(4)));  // (a slot's stride need not be a multiple of 16)

// A 16-token tile of one KV head as requested: 16 bytes of K and V of token lane / 4, and the scale of K (lanes 0..15) or
// V (16..31) of token lane % 16.
struct CacheTile {
  u32x4_t k, v;
  uint16_t scale;
};

__device__ __forceinline__ void request_tile(const ResidentArgs &a, uint32_t key_offset, uint32_t value_offset, const Run &run, uint32_t kv, uint32_t tile,
                                             uint32_t lane, CacheTile &out) {
  const uint32_t line = min(tile * kTile + (lane >> 2), run.length - 1), single = min(tile * kTile + (lane & 15), run.length - 1);
  const Global<uint8_t> row = global<uint8_t>(a.pool) + (size_t)run.slot(line) * a.token_stride + kv * 64 + (lane & 3) * 16;
  out.k = *(Global<cache_u32x4_t>)(row + key_offset);
  out.v = *(Global<cache_u32x4_t>)(row + value_offset);
  const uint32_t group = ((lane & 16 ? value_offset : key_offset) >> 6) + kv;
  out.scale = ((Global<uint16_t>)(global<uint8_t>(a.pool) + (size_t)run.slot(single) * a.token_stride + a.token_elements))[group];
}
// Rows of 64 bytes, their 16-byte pieces exchanged by the token / 4, which spreads the columns' reads over the banks.
__device__ __forceinline__ void keep_tile(uint8_t *patch, const CacheTile &tile, uint32_t lane) {
  const uint32_t token = lane >> 2, piece = (lane & 3) ^ (token >> 2);
  *reinterpret_cast<u32x4_t *>(patch + token * 64 + piece * 16) = tile.k;
  *reinterpret_cast<u32x4_t *>(patch + 1024 + token * 64 + piece * 16) = tile.v;
  if (lane < 32) reinterpret_cast<uint16_t *>(patch + 2048)[lane] = tile.scale;
}

// What a wave has of a run's attention: the running maximum of head lane % 16 (in base 2), its share of the denominator,
// and out[n][i]: column 4 (4 (lane / 16) + i) + n.
struct Attended {
  float top, sum;
  f4_t out[4];
};

// N 16-token tiles (of which tokens[] are there, of the first at least one) from their patches, in one step: the chain from
// the scores to the weights is longer than its instructions.  query: B operand of the score products; bias: what the
// biased decode of K adds to a head's scores.
template <int N>
__device__ __forceinline__ void walk_tiles(Attended &state, const uint8_t *patches, const h8_t (&query)[2], float bias, float score_scale,
                                           const uint32_t (&tokens)[N], uint32_t lane) {
  const uint32_t col = lane & 15, quad = lane >> 4;
  float score[N][4], most = state.top;
  uint32_t v[N][4];
  h2_t vs[N][2];
#pragma unroll
  for (int n = 0; n < N; ++n) {
    const uint8_t *patch = patches + n * kPatchBytes;
    const u32x4_t k = *reinterpret_cast<const u32x4_t *>(patch + col * 64 + (quad ^ (col >> 2)) * 16);
    const uint2 k_scale = *reinterpret_cast<const uint2 *>(patch + 2048 + quad * 8);
    const uint2 v_scale = *reinterpret_cast<const uint2 *>(patch + 2048 + 32 + quad * 8);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      v[n][i] = *reinterpret_cast<const uint32_t *>(patch + 1024 + (quad * 4 + i) * 64 + ((col >> 2) ^ quad) * 16 + (col & 3) * 4);
    f4_t part = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      h2_t h0, h1, h2, h3;
      int8x4_to_h2_biased(k[2 * j] ^ 0x80808080u, h0, h1);
      int8x4_to_h2_biased(k[2 * j + 1] ^ 0x80808080u, h2, h3);
      const h8_t key = {h0[0], h0[1], h1[0], h1[1], h2[0], h2[1], h3[0], h3[1]};
      part = __builtin_amdgcn_mfma_f32_16x16x32_f16(key, query[j], part, 0, 0, 0);
    }
    const h2_t ks[2] = {as_h2(k_scale.x), as_h2(k_scale.y)};
    vs[n][0] = as_h2(v_scale.x), vs[n][1] = as_h2(v_scale.y);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      score[n][i] = quad * 4 + i < tokens[n] ? (part[i] - bias) * (float)ks[i >> 1][i & 1] * score_scale : -INFINITY;
      most = fmaxf(most, score[n][i]);
    }
  }
  const float top = max_of_rows(most);  // (finite: the first token is there)
  const float alpha = __builtin_amdgcn_exp2f(state.top - top);
  state.top = top;
  float p[N][4], sum = 0.0f;
#pragma unroll
  for (int n = 0; n < N; ++n)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      p[n][i] = __builtin_amdgcn_exp2f(score[n][i] - top);
      sum += p[n][i];
    }
  state.sum = state.sum * alpha + sum;
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int i = 0; i < 4; ++i) state.out[c][i] *= alpha;
#pragma unroll
  for (int n = 0; n < N; ++n) {
    h4_t weight;
#pragma unroll
    for (int i = 0; i < 4; ++i) weight[i] = (_Float16)(p[n][i] * (float)vs[n][i >> 1][i & 1]);
    // four tokens x four columns -> four columns x four tokens
    const uint32_t a0 = v[n][0] ^ 0x80808080u, a1 = v[n][1] ^ 0x80808080u, a2 = v[n][2] ^ 0x80808080u, a3 = v[n][3] ^ 0x80808080u;
    const uint32_t t01_lo = __builtin_amdgcn_perm(a1, a0, 0x05010400u), t01_hi = __builtin_amdgcn_perm(a1, a0, 0x07030602u);
    const uint32_t t23_lo = __builtin_amdgcn_perm(a3, a2, 0x05010400u), t23_hi = __builtin_amdgcn_perm(a3, a2, 0x07030602u);
    const uint32_t columns[4] = {__builtin_amdgcn_perm(t23_lo, t01_lo, 0x05040100u), __builtin_amdgcn_perm(t23_lo, t01_lo, 0x07060302u),
                                 __builtin_amdgcn_perm(t23_hi, t01_hi, 0x05040100u), __builtin_amdgcn_perm(t23_hi, t01_hi, 0x07060302u)};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      h2_t lo, hi;
      int8x4_to_h2(columns[c], lo, hi);
      const h4_t values = {lo[0], lo[1], hi[0], hi[1]};
      state.out[c] = __builtin_amdgcn_mfma_f32_16x16x16f16(values, weight, state.out[c], 0, 0, 0);
    }
  }
}

// ---- the product phases ---------------------------------------------------------------------------------------
enum Product { kQkv = 0, kOut = 1, kGateUp = 2, kDown = 3 };
constexpr uint32_t kMostWidth = 1024, kMostMlp = 2048;  // of rows and of heads together; of the SwiGLU
constexpr int groups_most(int product) { return (product == kDown ? kMostMlp : kMostWidth) / 64 / kWaves; }  // of a wave: every eighth of the row's

// A wave's scale groups wave, wave + 8, ... of 16 weight rows, as a lane of the matrix instruction holds them (row lane % 16,
// K values [16 (lane / 16), + 16) of a group), and one of the tile's scales: of row t % 16 and group t / 16.
template <int G>
struct TileWeights {
  uint2 piece[G];
  uint16_t scale;
};

// ROTATED: of a rotated head's tile rows 8..15 are 32 columns on, the rotation's partners of rows 0..7.
template <bool ROTATED, int G>
__device__ __forceinline__ void request_weights(TileWeights<G> &out, uint32_t groups, Global<uint8_t> weight, Global<uint16_t> scale,
                                                uint32_t t, uint32_t wave) {
  const uint32_t row = (t & 15) + (ROTATED ? (t & 8) * 3 : 0), piece = row * groups * 32 + ((t >> 4) & 3) * 8 + wave * 32;
#pragma unroll
  for (int i = 0; i < G; ++i)
    if (wave + kWaves * i < groups) {
      const uint64_t bits = *(Global<uint64_t>)(weight + (piece + i * kWaves * 32));
      out.piece[i] = make_uint2((uint32_t)bits, (uint32_t)(bits >> 32));
    }
  out.scale = scale[row * groups + min(t >> 4, groups - 1)];
}

// This wave's share of a tile's 16 x 16 sums of N matrices over the same rows: lane (sequence lane % 16, columns
// 4 (lane / 16) + i).  x: the lane's part of the activations, of group `wave`.
template <int N, int G>
__device__ __forceinline__ void tile_share(f4_t (&sum)[N], const TileWeights<G> *const (&weights)[N], const uint16_t *scales, const uint16_t *x,
                                           uint32_t groups, uint32_t wave, uint32_t quad) {
#pragma unroll
  for (int n = 0; n < N; ++n) sum[n] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < G; ++i)
    if (wave + kWaves * i < groups) {  // (the same for the whole wave)
      const h8_t b[2] = {*reinterpret_cast<const h8_t *>(x + i * kWaves * 64), *reinterpret_cast<const h8_t *>(x + i * kWaves * 64 + 8)};
      uint2 scale[N];
      f4_t part[N];
#pragma unroll
      for (int n = 0; n < N; ++n) {
        scale[n] = *reinterpret_cast<const uint2 *>(scales + n * 16 * kTile + (wave + kWaves * i) * kTile + quad * 4);
        part[n] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
      }
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int n = 0; n < N; ++n) {
          const W4Pairs q = w4_decode_pairs(j == 0 ? weights[n]->piece[i].x : weights[n]->piece[i].y);
          const h8_t a = {q.p04[0], q.p04[1], q.p15[0], q.p15[1], q.p26[0], q.p26[1], q.p37[0], q.p37[1]};
          part[n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b[j], part[n], 0, 0, 0);
        }
#pragma unroll
      for (int n = 0; n < N; ++n) {
        const h2_t lo = as_h2(scale[n].x), hi = as_h2(scale[n].y);
        sum[n][0] += part[n][0] * (float)lo[0];
        sum[n][1] += part[n][1] * (float)lo[1];
        sum[n][2] += part[n][2] * (float)hi[0];
        sum[n][3] += part[n][3] * (float)hi[1];
      }
    }
}

// Runs that the workgroups of a launch can take: whole sets of the KV heads of eight.
__host__ __device__ __forceinline__ uint32_t resident_slots(uint32_t workgroups, uint32_t kv_heads) {
  return workgroups / (8 * kv_heads) * 8;
}

// ONE: one sequence.  All threads share its row, a word or two each; else a wave has a row.  TOGETHER: all the polling half's
// waves merge the runs of a (sequence, head); else a wave does, four runs a trip to memory, without a barrier.
template <bool ONE, bool TOGETHER>
struct Resident {
  static constexpr uint32_t kStep = ONE ? 1 : 2;  // cache tiles of a wave's step
  static constexpr uint32_t kSequenceStride = ONE ? kTile : kReduceStride, kWaveStride = ONE ? kTile : kTile * kReduceStride;
  const ResidentArgs &a;
  uint8_t *const lds;
  uint32_t t, lane, wave, quad;  // t, wave: within the half
  const uint32_t wg, workgroups;
  const uint32_t h, qd, kvd, mlp;
  const Run run;
  const Runs runs;
  const bool has_run, last_run;
  const uint32_t run_slot, kv_of_run;  // the run's place among all, and the KV head of it that the workgroup takes
  const uint32_t first_tag;  // of the first layer
  Patience patience;
  TileWeights<groups_most(kQkv)> w_qkv, w_out, w_gate, w_up;
  TileWeights<groups_most(kDown)> w_down;

  __device__ __forceinline__ const ResidentLayer &layer(uint32_t index) const {
    return reinterpret_cast<const ResidentLayer *>(lds + a.lds.layers)[index];
  }
  // What is computed from these is computed where it stands: the addresses are the same for every layer, and the compiler
  // would hold all of them, more than there are registers, from before the first.
  __device__ __forceinline__ void here() { asm volatile("" : "+v"(t), "+v"(lane), "+v"(quad)); }
  template <int P>
  __device__ __forceinline__ uint32_t depth() const { return P == kOut ? qd : P == kDown ? mlp : h; }

  template <int P>
  __device__ __forceinline__ void request(uint32_t index, uint32_t tile) {
    const ResidentLayer &of = layer(index);
    const auto at = [&](uint32_t which, uint32_t row) {
      const uint32_t groups = depth<P>() >> 6;
      const auto uniform = [](const void *pointer) {
        const uint64_t bits = reinterpret_cast<uint64_t>(pointer);
        return (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)bits) |
               (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(bits >> 32)) << 32;
      };
      const Global<uint8_t> weight = (Global<uint8_t>)uniform(of.weight[which]) + row * groups * 32;
      const Global<uint16_t> scale = (Global<uint16_t>)uniform(of.scale[which]) + row * groups;
      if constexpr (P == kQkv) request_weights<true>(w_qkv, groups, weight, scale, t, wave);
      if constexpr (P == kOut) request_weights<false>(w_out, groups, weight, scale, t, wave);
      if constexpr (P == kGateUp) {
        if (which == 4) request_weights<false>(w_gate, groups, weight, scale, t, wave);
        else request_weights<false>(w_up, groups, weight, scale, t, wave);
      }
      if constexpr (P == kDown) request_weights<false>(w_down, groups, weight, scale, t, wave);
    };
    if constexpr (P == kQkv) {
      const uint32_t head = tile >> 2, column = (tile & 3) * 8;
      const uint32_t which = head < a.q_heads ? 0 : head < a.q_heads + a.kv_heads ? 1 : 2;
      at(which, (head - (which == 0 ? 0 : which == 1 ? a.q_heads : a.q_heads + a.kv_heads)) * 64 + column);
    } else if constexpr (P == kGateUp) {
      at(4, tile * kTile);
      at(5, tile * kTile);
    } else {
      at(P == kOut ? 3 : 6, tile * kTile);
    }
  }

  // The rows of a product into LDS, normalised where it says so; a finishing thread's residual beside them.
  template <int P>
  __device__ __forceinline__ uint32_t stage(uint16_t *act, uint32_t row0, uint32_t rows, uint32_t tag, bool finishes, uint32_t residual_at) {
    constexpr bool kNorm = P == kQkv || P == kGateUp, kResidual = P == kOut || P == kDown;
    const uint32_t words = depth<P>() >> 1;
    const uint64_t *const hand = a.hand;
    const uint32_t from = a.words.in[P] + row0 * words, own_tag = P == kQkv ? tag - 1 : tag, residual_tag = P == kOut ? tag - 1 : tag;
    uint32_t residual = 0;
    if constexpr (ONE) {
      // (words: 512 at most, of the down projection 1024)
      constexpr int W = P == kDown ? 2 : 1, R = kResidual ? 1 : 0;
      uint64_t value[W + R];
      const bool present = wave * 64 < words;
      if (present) {
        uint32_t at[W + R], tags[W + R];
#pragma unroll
        for (int j = 0; j < W; ++j) {
          at[j] = from + min(t + j * kHalf, words - 1);
          tags[j] = own_tag;
        }
        if constexpr (R != 0) {
          at[W] = finishes ? residual_at : at[0];
          tags[W] = finishes ? residual_tag : own_tag;
        }
        await_words(value, hand, patience, at, tags);
        if constexpr (R != 0) residual = (uint32_t)value[W];
      }
      if constexpr (kNorm) {
        float *const squares = reinterpret_cast<float *>(lds + a.lds.squares);
        float square = 0.0f;
        if (present) {
          const h2_t x = as_h2((uint32_t)value[0]);
          square = wave_sum(t < words ? (float)x[0] * (float)x[0] + (float)x[1] * (float)x[1] : 0.0f);
        }
        if (lane == 0) squares[wave] = square;
        __syncthreads();
        const f4_t low = *reinterpret_cast<const f4_t *>(squares), high = *reinterpret_cast<const f4_t *>(squares + 4);
        const float total = ((low[0] + low[1]) + (low[2] + low[3])) + ((high[0] + high[1]) + (high[2] + high[3]));
        const float inverse = rsqrtf(total / (float)h + (P == kQkv ? a.attention_epsilon : a.ffn_epsilon));
        if (t < words) *reinterpret_cast<uint32_t *>(act + t * 2) = normalised<P>((uint32_t)value[0], t, inverse, gain_row(tag) + (P == kQkv ? 0 : h));
      } else {
#pragma unroll
        for (int j = 0; j < W; ++j)
          if (t + j * kHalf < words) *reinterpret_cast<uint32_t *>(act + (t + j * kHalf) * 2) = (uint32_t)value[j];
      }
      return residual;
    }
    if (kResidual && finishes) {
      uint64_t value[1];
      const uint32_t at[1] = {residual_at};
      await_words(value, hand, patience, at, residual_tag);
      residual = (uint32_t)value[0];
    }
    stage_row<P>(act, row0, rows, tag, wave);
    return residual;
  }

  // Several sequences, a wave's part (wave16: of both halves): a row to normalise, or its share of one as it is.
  template <int P>
  __device__ __forceinline__ void stage_row(uint16_t *act, uint32_t row0, uint32_t rows, uint32_t tag, uint32_t wave16) {
    constexpr bool kNorm = P == kQkv || P == kGateUp;
    const uint32_t words = depth<P>() >> 1, stride = depth<P>() + kRowPad, own_tag = P == kQkv ? tag - 1 : tag;
    const auto stage_words = [&](uint32_t row, uint32_t base, uint32_t step, auto width, auto use) {
      constexpr int W = decltype(width)::value;
      uint64_t value[W];
      const uint32_t from = a.words.in[P] + (row0 + row) * words;
      uint32_t at[W];
#pragma unroll
      for (int j = 0; j < W; ++j) at[j] = from + min(base + j * step + lane, words - 1);
      await_words(value, a.hand, patience, at, own_tag);
#pragma unroll
      for (int j = 0; j < W; ++j) use(j, base + j * step + lane, (uint32_t)value[j]);
    };
    if constexpr (kNorm) {  // 512 words at most
      if (wave16 >= rows) return;
      uint32_t *const to = reinterpret_cast<uint32_t *>(act + wave16 * stride);
      const uint16_t *const gain = gain_row(tag) + (P == kQkv ? 0 : h);
      uint32_t payload[8];
      float square = 0.0f;
      const auto take = [&](int j, uint32_t word, uint32_t bits) {
        payload[j] = bits;
        const h2_t x = as_h2(bits);
        if (word < words) square += (float)x[0] * (float)x[0] + (float)x[1] * (float)x[1];
      };
      if (words <= 256) stage_words(wave16, 0, 64, std::integral_constant<int, 4>(), take);
      else stage_words(wave16, 0, 64, std::integral_constant<int, 8>(), take);
      const float inverse = rsqrtf(wave_sum(square) / (float)h + (P == kQkv ? a.attention_epsilon : a.ffn_epsilon));
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (j * 64u < words && j * 64 + lane < words) to[j * 64 + lane] = normalised<P>(payload[j], j * 64 + lane, inverse, gain);
    } else {
      const uint32_t shift = rows <= 4 ? 2 : rows <= 8 ? 3 : 4, row = wave16 & ((1u << shift) - 1), part = wave16 >> shift, parts = 16u >> shift;
      if (row >= rows) return;
      uint32_t *const to = reinterpret_cast<uint32_t *>(act + row * stride);
#pragma unroll 1
      for (uint32_t base = part * 64; base < words; base += 6 * 64 * parts)
        stage_words(row, base, 64 * parts, std::integral_constant<int, 6>(), [&](int, uint32_t word, uint32_t bits) {
          if (word < words) to[word] = bits;
        });
    }
  }

  // The norm weights of a layer (its tag's): those of A, then those of E.
  __device__ __forceinline__ const uint16_t *gain_row(uint32_t tag) const {
    return reinterpret_cast<const uint16_t *>(lds + a.lds.gains) + ((tag - first_tag) & 1) * 2 * h;
  }
  template <int P>
  __device__ __forceinline__ uint32_t normalised(uint32_t payload, uint32_t word, float inverse, const uint16_t *gain) const {
    const h2_t x = as_h2(payload);
    const uint32_t column = word_column(word);
    const float g0 = half_bits_to_float(gain[column]), g1 = half_bits_to_float(gain[column + 4]);
    return P == kGateUp ? two_halves((float)x[0] * g0 * inverse, (float)x[1] * g1 * inverse)
                        : two_halves((float)x[0] * inverse * g0, (float)x[1] * inverse * g1);
  }

  __device__ __forceinline__ void leave(float *reduce, f4_t sum) const {
    if (!ONE || (lane & 15) == 0) *reinterpret_cast<f4_t *>(reduce + wave * kWaveStride + (lane & 15) * kSequenceStride + quad * 4) = sum;
  }
  __device__ __forceinline__ float whole(const float *reduce, uint32_t sequence, uint32_t column) const {
    float part[kWaves];
#pragma unroll
    for (uint32_t w = 0; w < kWaves; ++w) part[w] = reduce[w * kWaveStride + sequence * kSequenceStride + column];
    return ((part[0] + part[1]) + (part[2] + part[3])) + ((part[4] + part[5]) + (part[6] + part[7]));
  }

  // A, D, E or F of a layer.  The next layer's weights are requested when the words are out: they land while those travel.
  template <int P>
  __device__ __forceinline__ void product(uint32_t index, uint32_t next, bool last, uint32_t tag) {
    const uint32_t groups = depth<P>() >> 6, stride = depth<P>() + kRowPad;
    uint16_t *const act = reinterpret_cast<uint16_t *>(lds);
    float *const reduce = reinterpret_cast<float *>(lds + a.lds.reduce);
    uint16_t *const scales = reinterpret_cast<uint16_t *>(lds + a.lds.scales);
    const uint32_t units = a.units[P], tiles = a.tiles[P];
#pragma unroll 1
    for (uint32_t unit = wg; unit < units; unit = ONE ? units : unit + workgroups) {  // (one sequence: a unit a workgroup at most)
      const uint32_t group = ONE ? 0 : unit / tiles, tile = ONE ? unit : unit - group * tiles, row0 = group * a.unit_rows[P];
      const uint32_t rows = ONE ? 1 : min(a.unit_rows[P], a.m - row0);
      if (!ONE && unit != wg) request<P>(index, tile);
      // a thread of the epilogue finishes one column of one sequence
      const uint32_t column = t & 15, local = ONE ? 0 : min(t >> 4, rows - 1), sequence = row0 + local;
      const uint32_t word = tile * 8 + (column >> 3) * 4 + (column & 3);  // of the product's row, columns `column` and + 4
      const bool finishes = t < rows * 16;
      const uint32_t of_head = (tile & 3) * 8 + (column & 7) + (column & 8) * 4;  // (of QKV)
      uint16_t cosine = 0, sine = 0;
      if (P == kQkv && finishes) {
        cosine = a.cosine[sequence * 64 + of_head];
        sine = a.sine[sequence * 64 + of_head];
      }
      const uint32_t residual = stage<P>(act, row0, rows, tag, finishes, (P == kOut ? a.words.x : a.words.mid) + sequence * (h >> 1) + word);
      if (t < groups * kTile) {  // [group][row]
        if constexpr (P == kQkv) scales[t] = w_qkv.scale;
        if constexpr (P == kOut) scales[t] = w_out.scale;
        if constexpr (P == kGateUp) {
          scales[t] = w_gate.scale;
          scales[16 * kTile + t] = w_up.scale;
        }
        if constexpr (P == kDown) scales[t] = w_down.scale;
      }
      __syncthreads();
      const uint16_t *const x = act + (ONE ? 0 : min(lane & 15, rows - 1) * stride) + quad * 16 + wave * 64;
      f4_t sum[P == kGateUp ? 2 : 1];
      if constexpr (P == kGateUp) {
        const TileWeights<groups_most(P)> *const both[2] = {&w_gate, &w_up};
        tile_share<2, groups_most(P)>(sum, both, scales, x, groups, wave, quad);
        leave(reduce + kReduceWords, sum[1]);
      } else if constexpr (P == kDown) {
        const TileWeights<groups_most(P)> *const one[1] = {&w_down};
        tile_share<1, groups_most(P)>(sum, one, scales, x, groups, wave, quad);
      } else {
        const TileWeights<groups_most(P)> *const one[1] = {P == kQkv ? &w_qkv : &w_out};
        tile_share<1, groups_most(P)>(sum, one, scales, x, groups, wave, quad);
      }
      leave(reduce, sum[0]);
      __syncthreads();
      if (finishes) {
        const float own = whole(reduce, local, column);
        if constexpr (P == kQkv) {
          const _Float16 value = (_Float16)own, partner = (_Float16)moved<kFromEighth>(own);
          const uint32_t head = tile >> 2;
          const _Float16 out = head < a.q_heads + a.kv_heads
                                   ? rotate_half_value(value, partner, __builtin_bit_cast(_Float16, cosine), __builtin_bit_cast(_Float16, sine), column < 8)
                                   : value;
          const float beside = moved<kFromNext>((float)out);
          if ((column & 1) == 0)
            hand_store(a.hand, a.words.qkv + sequence * ((qd + 2 * kvd) >> 1) + head * 32 + (of_head >> 1), two_halves((float)out, beside), tag);
        } else {
          float value = own;
          if constexpr (P == kGateUp) {
            value = own / (1.0f + __expf(-own)) * whole(reduce + kReduceWords, local, column);
          } else {
            const h2_t x2 = as_h2(residual);
            value += (float)((column & 4) == 0 ? x2[0] : x2[1]);
          }
          const float fourth = moved<kFromFourth>(value);
          if ((column & 4) == 0) {
            const uint32_t bits = two_halves(value, fourth);
            if (P == kDown && last) {
              uint16_t *to = a.x_out + sequence * h + word_column(word);
              to[0] = (uint16_t)bits;
              to[4] = (uint16_t)(bits >> 16);
            } else {
              hand_store(a.hand, a.words.out[P] + sequence * (P == kGateUp ? mlp >> 1 : h >> 1) + word, bits, tag);
            }
          }
        }
      }
    }
    if (wg < units) request<P>(next, ONE ? wg : wg % tiles);
    asm volatile("" ::: "memory");  // (the requests stay here)
  }

  // B's end: the waves' shares of a run and, of a sequence's last one, its new token; a head a wave, both halves' waves.
  __device__ __forceinline__ void hand_run(uint32_t tag, uint32_t wave16) {
    const uint32_t per_kv = a.per_kv;
    if (wave16 >= per_kv) return;
    const uint32_t head = kv_of_run * per_kv + wave16;
    const float *const run_out = reinterpret_cast<const float *>(lds + a.lds.run_out) + wave16 * kRunStride;
    const uint32_t next = per_kv * kRunStride;  // (to the next wave's)
    float fresh = -INFINITY, fresh_value = 0.0f;
    if (last_run) {
      fresh = reinterpret_cast<const float *>(lds + a.lds.new_score)[head];
      fresh_value = half_bits_to_float(reinterpret_cast<const uint16_t *>(lds + a.lds.new_rows)[qd + kvd + kv_of_run * 64 + lane]);
    }
    // lane s % 8: maximum and sum of the s-th wave
    const uint32_t own = (lane & 7) * next;
    const float own_top = run_out[own + 64], own_sum = run_out[own + 65];
    float part[kWaves];
#pragma unroll
    for (uint32_t s = 0; s < kWaves; ++s) part[s] = run_out[s * next + lane];
    float top = own_top;
    top = fmaxf(top, moved<0xB1>(top));
    top = fmaxf(top, moved<0x4E>(top));
    top = fmaxf(fmaxf(top, moved<0x141>(top)), fresh);
    const float own_weight = __builtin_amdgcn_exp2f(own_top - top);  // (0 where the wave had no tokens)
    float sum = own_sum * own_weight;
    sum += moved<0xB1>(sum);
    sum += moved<0x4E>(sum);
    sum += moved<0x141>(sum);
    float value = 0.0f;
#pragma unroll
    for (uint32_t s = 0; s < kWaves; ++s)
      value += part[s] * __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, own_weight), s));
    if (last_run) {
      const float weight = __builtin_amdgcn_exp2f(fresh - top);
      sum += weight;
      value += fresh_value * weight;
    }
    const uint32_t out = a.words.parts + (run_slot * a.q_heads + head) * kPartWords;
    hand_store(a.hand, out + lane, __builtin_bit_cast(uint32_t, value / sum), tag);
    if (lane == 0) hand_store(a.hand, out + 64, __builtin_bit_cast(uint32_t, top + __builtin_amdgcn_logf(sum)), tag);
  }

  // B, the polling half's part.
  __device__ __forceinline__ void hand_queries(uint32_t tag) {
    uint32_t *const new_rows = reinterpret_cast<uint32_t *>(lds + a.lds.new_rows);
    const uint32_t from = a.words.qkv + run.sequence * ((qd + 2 * kvd) >> 1);
    // of the workgroup's KV head: the queries, the key, the value (at most 576 words)
    const uint32_t q_words = a.per_kv * 32, wanted = q_words + 64;
#pragma unroll 1
    for (uint32_t base = 0; base < wanted; base += kHalf) {
      const uint32_t own = base + t, past = own - q_words;
      const uint32_t word = own < q_words ? kv_of_run * q_words + own : (qd >> 1) + kv_of_run * 32 + (past & 31) + (past >> 5) * (kvd >> 1);
      if (own < wanted) {
        uint64_t value[1];
        const uint32_t at[1] = {from + word};
        await_words(value, a.hand, patience, at, tag);
        new_rows[word] = (uint32_t)value[0];
      }
    }
    __syncthreads();
    if (last_run) {  // the new token's scores
      const uint16_t *const rows = reinterpret_cast<const uint16_t *>(new_rows);
      for (uint32_t head = kv_of_run * a.per_kv + wave; head < (kv_of_run + 1) * a.per_kv; head += kWaves) {
        const float score = wave_sum(half_bits_to_float(rows[head * 64 + lane]) * half_bits_to_float(rows[qd + head / a.per_kv * 64 + lane])) *
                            (a.scale * 1.4426950408889634f);
        if (lane == 0) reinterpret_cast<float *>(lds + a.lds.new_score)[head] = score;
      }
    }
    __syncthreads();
    hand_run(tag, wave);
  }

  // C: the runs of a (sequence, head) together.
  __device__ __forceinline__ void merge(uint32_t tag) {
    constexpr uint32_t share = TOGETHER ? kWaves : 1;
    const uint32_t all = a.m * a.q_heads;
#pragma unroll 1
    for (uint32_t unit = TOGETHER ? wg : wg + wave * workgroups; unit < all; unit = TOGETHER ? all : unit + kWaves * workgroups) {
      const uint32_t sequence = ONE ? 0 : unit / a.q_heads, head = unit - sequence * a.q_heads;
      const uint32_t first = (uint32_t)__builtin_amdgcn_readlane((int)runs.first, (int)sequence);
      const uint32_t count = (uint32_t)__builtin_amdgcn_readlane((int)runs.count, (int)sequence);
      const uint32_t from = a.words.parts + (first * a.q_heads + head) * kPartWords, step = a.q_heads * kPartWords;
      float top = -INFINITY, sum = 0.0f, value = 0.0f;
#pragma unroll 1
      for (uint32_t run0 = TOGETHER ? wave : 0; run0 < count; run0 += 4 * share) {
        // four runs: their values, and in lane j % 4 the weight of the j-th (of runs beyond the last: that one's, not used)
        uint64_t word[5];
        uint32_t at[5];
#pragma unroll
        for (int j = 0; j < 5; ++j) at[j] = from + min(run0 + (j < 4 ? j : lane & 3) * share, count - 1) * step + (j < 4 ? lane : 64);
        await_words(word, a.hand, patience, at, tag);
        const bool there = run0 + (lane & 3) * share < count;
        const float weight_log = there ? __builtin_bit_cast(float, (uint32_t)word[4]) : -INFINITY;
        float most = weight_log;  // over the four
        most = fmaxf(most, moved<0xB1>(most));
        most = fmaxf(most, moved<0x4E>(most));
        most = fmaxf(most, top);
        const float old = __builtin_amdgcn_exp2f(top - most), own = __builtin_amdgcn_exp2f(weight_log - most);
        top = most;
        sum *= old;
        value *= old;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float weight = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, own), j));
          sum += weight;
          value += run0 + j * share < count ? weight * __builtin_bit_cast(float, (uint32_t)word[j]) : 0.0f;
        }
      }
      if constexpr (TOGETHER) {
        float *const shares = reinterpret_cast<float *>(lds + a.lds.merge);
        shares[wave * 64 + lane] = value;
        if (lane == 0) {
          shares[kWaves * 64 + wave] = top;
          shares[kWaves * 65 + wave] = sum;
        }
        __syncthreads();
        if (wave != 0) return;
        float tops[kWaves];
#pragma unroll
        for (uint32_t w = 0; w < kWaves; ++w) tops[w] = shares[kWaves * 64 + w];
        top = tops[0];
#pragma unroll
        for (uint32_t w = 1; w < kWaves; ++w) top = fmaxf(top, tops[w]);
        sum = value = 0.0f;
#pragma unroll
        for (uint32_t w = 0; w < kWaves; ++w) {
          const float weight = __builtin_amdgcn_exp2f(tops[w] - top);
          sum += weight * shares[kWaves * 65 + w];
          value += weight * shares[w * 64 + lane];
        }
      }
      value /= sum;
      const float partner = moved<kFromFourth>(value);
      if ((lane & 4) == 0)
        hand_store(a.hand, a.words.attention + sequence * (qd >> 1) + head * 32 + (lane >> 3) * 4 + (lane & 3), two_halves(value, partner), tag);
    }
  }

  __device__ __forceinline__ void poll_and_multiply(uint32_t base_tag, uint32_t layer_count) {
    const auto first = [&](uint32_t product) { return ONE ? wg : wg % a.tiles[product]; };
    if (wg < a.units[kQkv]) request<kQkv>(0, first(kQkv));
    if (wg < a.units[kOut]) request<kOut>(0, first(kOut));
    if (wg < a.units[kGateUp]) request<kGateUp>(0, first(kGateUp));
    if (wg < a.units[kDown]) request<kDown>(0, first(kDown));
    // the rows that come in, as the words that a layer in front of the first would have left
    for (uint32_t unit = wg; unit < a.units[kDown]; unit += workgroups) {
      const uint32_t group = ONE ? 0 : unit / a.tiles[kDown], tile = unit - group * a.tiles[kDown], row0 = group * a.unit_rows[kDown];
      const uint32_t sequence = row0 + (t >> 3), word = tile * 8 + (t & 7), column = word_column(word);
      if (t < min(a.unit_rows[kDown], a.m - row0) * 8)
        hand_store(a.hand, a.words.x + sequence * (h >> 1) + word,
                   (uint32_t)a.x_in[sequence * h + column] | (uint32_t)a.x_in[sequence * h + column + 4] << 16, base_tag);
    }
#pragma unroll 1
    for (uint32_t index = 0; index < layer_count; ++index) {
      const bool last = index + 1 == layer_count;
      const uint32_t next = last ? index : index + 1, tag = base_tag + 1 + index;
      here();
      if (!ONE) __syncthreads();  // (the norm weights; one sequence's norm has a barrier in front of them)
      product<kQkv>(index, next, last, tag);
      if (has_run) hand_queries(tag);
      merge(tag);
      product<kOut>(index, next, last, tag);
      product<kGateUp>(index, next, last, tag);
      product<kDown>(index, next, last, tag);
    }
  }

  // The other half: the cache, the norm weights, and the other half's barriers - per layer one, then those of its products,
  // its run and its merges.
  __device__ __forceinline__ void walk_cache(uint32_t base_tag, uint32_t layer_count) {
    const uint32_t tiles = (run.length + kTile - 1) / kTile, per_kv = a.per_kv;
    const bool walks = wave < tiles;
    uint8_t *const patch = lds + a.lds.patches + wave * (kStep * kPatchBytes);
    const uint16_t *const new_rows = reinterpret_cast<const uint16_t *>(lds + a.lds.new_rows);
    const uint32_t new_slot = last_run ? a.new_slots[run.sequence] : 0;
    // steps of kStep tiles: one step's in the wave's patches, the next one's on their way into registers
    CacheTile ahead[kStep];
    const auto has_step = [&](uint32_t step) { return walks && wave + kStep * step * kWaves < tiles; };
    const auto request_step = [&](uint32_t index, uint32_t step) {
      if (!has_step(step)) return;
      const ResidentLayer &of = layer(index);
      const uint32_t key_offset = of.key_offset, value_offset = of.value_offset;
#pragma unroll
      for (uint32_t n = 0; n < kStep; ++n)
        request_tile(a, key_offset, value_offset, run, kv_of_run, wave + (kStep * step + n) * kWaves, lane, ahead[n]);
    };
    const auto keep_step = [&](uint32_t step) {
      if (!has_step(step)) return;
#pragma unroll
      for (uint32_t n = 0; n < kStep; ++n) keep_tile(patch + n * kPatchBytes, ahead[n], lane);
    };
    uint16_t gain_bits[2][2];
    const auto request_gains = [&](uint32_t index) {
      const ResidentLayer &of = layer(index);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        gain_bits[0][i] = global<uint16_t>(of.attention_norm)[min(t + i * kHalf, h - 1)];
        gain_bits[1][i] = global<uint16_t>(of.ffn_norm)[min(t + i * kHalf, h - 1)];
      }
    };
    request_step(0, 0);
    keep_step(0);
    request_step(0, 1);
#pragma unroll 1
    for (uint32_t index = 0; index < layer_count; ++index) {
      const uint32_t next = min(index + 1, layer_count - 1), tag = base_tag + 1 + index;
      here();
      if (!ONE) __syncthreads();
      request_gains(next);
      other_half<kQkv>(tag);
      if (has_run) {
        __syncthreads();
        {
          const uint32_t col = lane & 15;
          const float score_scale = a.scale * 1.4426950408889634f;
          h8_t query[2];
          float bias = 0.0f;
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const uint4 bits = *reinterpret_cast<const uint4 *>(new_rows + (kv_of_run * per_kv + min(col, per_kv - 1)) * 64 + quad * 16 + j * 8);
            query[j] = __builtin_bit_cast(h8_t, col < per_kv ? bits : make_uint4(0, 0, 0, 0));
            const h2_t ones = {(_Float16)1.0f, (_Float16)1.0f};
            bias = __builtin_amdgcn_fdot2(as_h2(col < per_kv ? bits.x : 0), ones, bias, false);
            bias = __builtin_amdgcn_fdot2(as_h2(col < per_kv ? bits.y : 0), ones, bias, false);
            bias = __builtin_amdgcn_fdot2(as_h2(col < per_kv ? bits.z : 0), ones, bias, false);
            bias = __builtin_amdgcn_fdot2(as_h2(col < per_kv ? bits.w : 0), ones, bias, false);
          }
          bias = 1152.0f * sum_of_rows(bias);
          Attended state = {-INFINITY, 0.0f, {}};
#pragma unroll 1
          for (uint32_t step = 0; has_step(step); ++step) {
            uint32_t tokens[kStep];
#pragma unroll
            for (uint32_t n = 0; n < kStep; ++n) {
              const uint32_t first = (wave + (kStep * step + n) * kWaves) * kTile;
              tokens[n] = first < run.length ? run.length - first : 0;
            }
            __builtin_amdgcn_wave_barrier();
            walk_tiles<kStep>(state, patch, query, bias, score_scale, tokens, lane);
            __builtin_amdgcn_wave_barrier();
            keep_step(step + 1);
            request_step(index, step + 2);
          }
          state.sum = sum_of_rows(state.sum);
          if (col < per_kv) {  // (tokens or not: hand_run reads all)
            float *row = reinterpret_cast<float *>(lds + a.lds.run_out) + (wave * per_kv + col) * kRunStride;
#pragma unroll
            for (int i = 0; i < 4; ++i)
              *reinterpret_cast<f4_t *>(row + 4 * (quad * 4 + i)) = f4_t{state.out[0][i], state.out[1][i], state.out[2][i], state.out[3][i]};
            if (quad == 0) {
              row[64] = state.top;
              row[65] = state.sum;
            }
          }
        }
        __syncthreads();
        hand_run(tag, kWaves + wave);
        if (last_run) {  // the new token's slot: a group of 64 values a wave
          const ResidentLayer &of = layer(index);
          if (const uint32_t group = kv_of_run + wave * a.kv_heads; wave < 2) {  // K, V
            const uint32_t own = group < a.kv_heads ? group : group - a.kv_heads;
            const uint32_t segment = (group < a.kv_heads ? of.key_offset : of.value_offset) + own * 64;
            uint8_t *token = a.pool + (size_t)new_slot * a.token_stride;
            uint16_t stored;
            reinterpret_cast<int8_t *>(token)[segment + lane] = q8_quantize(half_bits_to_float(new_rows[qd + group * 64 + lane]), &stored);
            if (lane == 0) reinterpret_cast<uint16_t *>(token + a.token_elements)[segment >> 6] = stored;
          }
        }
        request_step(next, 0);
        asm volatile("" ::: "memory");
      }
      uint16_t *const gains = const_cast<uint16_t *>(gain_row(tag + 1));
#pragma unroll
      for (int i = 0; i < 2; ++i)
        if (t + i * kHalf < h) {
          gains[t + i * kHalf] = gain_bits[0][i];
          gains[h + t + i * kHalf] = gain_bits[1][i];
        }
      if (TOGETHER && wg < a.m * a.q_heads) __syncthreads();
      other_half<kOut>(tag);
      other_half<kGateUp>(tag);
      keep_step(0);  // (there by now)
      request_step(next, 1);
      asm volatile("" ::: "memory");
      other_half<kDown>(tag);
    }
  }

  // A product, the walking half's part: its barriers, and some of the rows of several sequences.
  template <int P>
  __device__ __forceinline__ void other_half(uint32_t tag) {
#pragma unroll 1
    for (uint32_t unit = wg; unit < a.units[P]; unit = ONE ? a.units[P] : unit + workgroups) {
      if (ONE) {
        if (P == kQkv || P == kGateUp) __syncthreads();
      } else {
        const uint32_t row0 = unit / a.tiles[P] * a.unit_rows[P];
        stage_row<P>(reinterpret_cast<uint16_t *>(lds), row0, min(a.unit_rows[P], a.m - row0), tag, kWaves + wave);
      }
      __syncthreads();
      __syncthreads();
    }
  }
};

template <bool ONE, bool TOGETHER>
__global__ __launch_bounds__(kThreads) void decode_resident_kernel(ResidentArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t resident_lds[];
  const uint32_t wg = blockIdx.x, wave16 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), t = threadIdx.x & (kHalf - 1);
  const uint32_t base_tag = *a.tag;
  for (uint32_t i = threadIdx.x; i < a.layer_count * (uint32_t)(sizeof(ResidentLayer) / 4); i += kThreads)
    reinterpret_cast<uint32_t *>(resident_lds + a.lds.layers)[i] = reinterpret_cast<const uint32_t *>(a.layers)[i];
  // A run's KV heads go to workgroups eight apart: on one XCD, whose L2 then serves all of them the lines that they share.
  const uint32_t band = 8 * a.kv_heads, run_slot = wg / band * 8 + wg % 8, slots = resident_slots(gridDim.x, a.kv_heads);
  const Runs runs = deal_runs(a, slots, 4 * kTile);
  const uint64_t mine = __builtin_amdgcn_ballot_w64(run_slot >= runs.first && run_slot < runs.first + runs.count);
  const bool has_run = mine != 0;
  const int owner = has_run ? __builtin_ctzll(mine) : 0;
  const uint32_t first = (uint32_t)__builtin_amdgcn_readlane((int)runs.first, owner);
  const uint32_t tokens = (uint32_t)__builtin_amdgcn_readlane((int)runs.tokens, owner);
  const uint32_t past = (uint32_t)__builtin_amdgcn_readlane((int)runs.past, owner);
  const uint32_t begin = has_run ? min((run_slot - first) * tokens, past) : 0;
  const bool last_run = has_run && run_slot - first + 1 == (uint32_t)__builtin_amdgcn_readlane((int)runs.count, owner);
  uint32_t *slot_cache = reinterpret_cast<uint32_t *>(resident_lds + a.lds.slots);
  const Run run = {(uint32_t)owner, has_run ? min(tokens, past - begin) : 0,
                   global<uint32_t>(a.slots + (uint32_t)__builtin_amdgcn_readlane((int)runs.offset, owner) + begin), (Local<uint32_t>)slot_cache};
  // Launches pack the new tokens of all sequences before any of them reads the cache; here the cache is read layers ahead.  So a
  // step in which a sequence reads a slot that the step itself writes (consecutive tokens of one sequence as rows of a batch) is left
  // to them.
  const uint32_t t64 = threadIdx.x & 63, new_slot = t64 < a.m ? a.new_slots[t64] : 0;
  bool written_now = false;
  for (uint32_t i = threadIdx.x; i < run.length; i += kThreads) {
    const uint32_t slot = run.slots[i];
    if (i < kSlotCache) slot_cache[i] = slot;
    for (uint32_t s = 0; s < a.m; ++s) written_now |= slot == (uint32_t)__builtin_amdgcn_readlane((int)new_slot, (int)s);
  }
  if (written_now) __hip_atomic_store(a.failed, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (threadIdx.x < a.h) {
    uint16_t *const gains = reinterpret_cast<uint16_t *>(resident_lds + a.lds.gains);
    gains[threadIdx.x] = a.layers[0].attention_norm[threadIdx.x];
    gains[a.h + threadIdx.x] = a.layers[0].ffn_norm[threadIdx.x];
  }
  __syncthreads();
  const uint32_t qd = a.q_heads * 64;
  Resident<ONE, TOGETHER> resident = {a, resident_lds, t, t & 63, wave16 & (kWaves - 1), (t & 63) >> 4, wg, gridDim.x, a.h, qd, a.kv_heads * 64, a.mlp,
                            run, runs, has_run, last_run, run_slot, wg % band / 8, base_tag + 1,
                            Patience{a.failed, a.wait_ticks, false}, {}, {}, {}, {}, {}};
  if (wave16 < kWaves)
    resident.poll_and_multiply(base_tag, a.layer_count);
  else
    resident.walk_cache(base_tag, a.layer_count);
}

uint32_t padded(uint32_t bytes) { return (bytes + 15) & ~15u; }

}  // namespace

bool resident_ok(uint32_t m, uint32_t h, uint32_t q_heads, uint32_t kv_heads, uint32_t mlp, uint32_t layers) {
  return m >= 1 && m <= kResidentRows && layers >= 1 && layers <= kResidentLayers && h % 64 == 0 && h >= 64 && h <= kMostWidth && kv_heads >= 1 &&
         kv_heads <= 8 && q_heads >= 1 && q_heads * 64 <= kMostWidth && q_heads % kv_heads == 0 && mlp % 64 == 0 && mlp >= 64 && mlp <= kMostMlp;
}

// Workgroups: one a CU at most, so that all are resident together.  One sequence takes as many as its widest phase has tiles, the
// fewest with which no workgroup has two (96 for 1536 columns of gate and up; with 96 / 128 / 192 / 256, 30 layers take 348 / 347 /
// 348 / 353 us behind 512 tokens, 361 / 355 / 354 / 354 behind 2048, 399 / 406 / 394 / 408 behind 8192: no count is steadily faster,
// and the rest of the chip stays free).  Several sequences take all CUs for the cache.
uint32_t resident_workgroups(uint32_t m, uint32_t h, uint32_t q_heads, uint32_t kv_heads, uint32_t mlp, uint32_t compute_units) {
  const uint32_t tiles_m = (m + kTile - 1) / kTile;
  const uint32_t widest = std::max(std::max((q_heads + 2 * kv_heads) * 4, mlp / kTile), h / kTile) * tiles_m;
  return m == 1 ? widest : std::min(compute_units, 256u);  // (one sequence: no workgroup has two tiles of a product)
}

ResidentWords resident_words(uint32_t m, uint32_t h, uint32_t q_heads, uint32_t kv_heads, uint32_t mlp, uint32_t workgroups) {
  ResidentWords words = {};
  uint32_t at = 0;
  auto take = [&](uint32_t count) {
    const uint32_t first = at;
    at += (count + 15) & ~15u;
    return first;
  };
  words.x = take(m * (h / 2));
  words.mid = take(m * (h / 2));
  words.qkv = take(m * (q_heads + 2 * kv_heads) * 32);
  words.attention = take(m * q_heads * 32);
  words.product = take(m * (mlp / 2));
  words.parts = take(workgroups * q_heads * kPartWords);
  words.total = at;
  words.in[0] = words.x, words.in[1] = words.attention, words.in[2] = words.mid, words.in[3] = words.product;
  words.out[0] = words.qkv, words.out[1] = words.mid, words.out[2] = words.product, words.out[3] = words.x;
  return words;
}

// Lays out a workgroup's memory and deals the products to the workgroups: units of as few sequences (four, eight or
// sixteen) as still leave each workgroup at most one: fewer words for each to poll.
uint32_t resident_lds(ResidentArgs &a, uint32_t workgroups) {
  const uint32_t qd = a.q_heads * 64, kvd = a.kv_heads * 64;
  const uint32_t k[4] = {a.h, qd, a.h, a.mlp}, tiles[4] = {(qd + 2 * kvd) / kTile, a.h / kTile, a.mlp / kTile, a.h / kTile};
  uint32_t at = 0;
  for (int p = 0; p < 4; ++p) {
    uint32_t rows = kTile;
    while (rows > 4 && tiles[p] * ((a.m + rows / 2 - 1) / (rows / 2)) <= workgroups) rows /= 2;
    a.unit_rows[p] = std::min(rows, a.m);
    a.tiles[p] = tiles[p];
    a.units[p] = tiles[p] * ((a.m + rows - 1) / rows);
    at = std::max(at, padded(a.unit_rows[p] * (k[p] + kRowPad) * 2));
  }
  const auto take = [&](uint32_t bytes) {
    const uint32_t first = at;
    at += padded(bytes);
    return first;
  };
  a.lds.new_rows = take((qd + 2 * kvd) * 2);
  a.lds.new_score = take(a.q_heads * 4);
  a.lds.run_out = take(kWaves * a.per_kv * kRunStride * 4);
  a.lds.reduce = take(2 * kReduceWords * 4);
  a.lds.scales = take(32 * kTile * 2);
  a.lds.gains = take(2 * 2 * a.h * 2);
  a.lds.squares = take(kWaves * 4);
  a.lds.patches = take(kWaves * 2 * kPatchBytes);
  a.lds.slots = take(kSlotCache * 4);
  a.lds.layers = take(a.layer_count * (uint32_t)sizeof(ResidentLayer));
  a.lds.merge = take(kWaves * 66 * 4);
  return at;
}

bool resident_fits(const ResidentArgs &args, uint32_t workgroups, uint32_t lds) {
  return lds <= kLdsMost && resident_slots(workgroups, args.kv_heads) >= args.m && workgroups <= (uint32_t)device_compute_units();
}

template <bool ONE, bool TOGETHER>
hipError_t launch_instance(const ResidentArgs &args, uint32_t workgroups, uint32_t lds, hipStream_t stream) {
  static bool configured[kMaxDevices] = {};
  if (hipError_t status = allow_dynamic_lds(reinterpret_cast<const void *>(decode_resident_kernel<ONE, TOGETHER>), kLdsMost, configured))
    return status;
  hipLaunchKernelGGL((decode_resident_kernel<ONE, TOGETHER>), dim3(workgroups), dim3(kThreads), lds, stream, args);
  return hipGetLastError();
}

hipError_t launch_decode_resident(const ResidentArgs &args, uint32_t workgroups, uint32_t lds, hipStream_t stream) {
  if (!resident_fits(args, workgroups, lds)) return hipErrorInvalidValue;
  if (args.m == 1) return launch_instance<true, true>(args, workgroups, lds, stream);  // (a workgroup a query head and more)
  // Sixteen runs a sequence and more: four trips of one wave.  us a step, one wave / eight: 2 sequences 442 / 475 behind 512 tokens,
  // 552 / 481 behind 2048, 641 / 515 behind 8192; 4 sequences 483 / 508, 573 / 527, 618 / 590; 8 (ten runs) 486 / 516, 518 / 536, 706 / 734.
  const bool together = resident_slots(workgroups, args.kv_heads) >= 16 * args.m && args.m * args.q_heads <= workgroups;
  return together ? launch_instance<false, true>(args, workgroups, lds, stream) : launch_instance<false, false>(args, workgroups, lds, stream);
}

}  // namespace llmopt
