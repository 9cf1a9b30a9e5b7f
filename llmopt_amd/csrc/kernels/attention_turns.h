// Attention of a prompt's rows by two groups of waves that take turns at the matrix cores (dense_attention.hip,
// chunk_attention.hip).
//
// A workgroup is eight waves, two on each SIMD, over the rows of one head, 32 a wave.  A wave's step is
//
//   weights    the next copies asked for, then the softmax of its scores of 64 keys
//   products   S^T of its next 64 keys = K Q^T, and O^T += V^T P^T of those weights
//
// with a barrier behind each, and group 1 (waves 4 .. 7) is one barrier behind group 0, so that while one wave of a SIMD has
// the matrix core the other has the vector unit.  Waves that were left to themselves did both one after the other: at 32 x 32
// tiles of heads of 128 the products, the reads of K and V from LDS and the softmax take about as long as each other, and a step
// took their sum.  The older wave of a SIMD wins where both want to issue: group 1's products go with a higher priority (products of
// heads of 128 in fp16 take 1535 cycles in both groups then; 1890 in group 1 and 1250 in group 0 without).
//
//  * SPLIT: both groups own the same 128 rows and take alternate stages of 64 keys, each through two stages of its own in LDS;
//    group 0 has both shares in the end.  Else 256 rows, and both groups read the same three stages.
//  * S^T leaves lane (j = lane % 32, half = lane / 32) sixteen scores of query row j for every 32 keys, keys
//    (r / 4) * 8 + half * 4 + r % 4, which are the B operand of O^T: weights never leave their lane.
//  * K and V go global -> LDS as 16-byte pieces that pass no registers, K's XOR-ed by the key, V's by twice the key (the
//    transposing reads of V take four rows at a time).
//  * V of step s + 1 and K of step s + 2 are asked for with weights s, when the last reads of what they replace lie behind a
//    barrier, and are first read with products s + 1, a step later.  Group 0 (SPLIT: both) waits for them at the end of
//    weights s + 1, where the copies asked for in between may still be under way; group 1 of the shared stages, a barrier later,
//    at the end of its products s.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "dense_attention_rule.h"
#include "staggered.h"

namespace llmopt {

typedef float f32x16 __attribute__((ext_vector_type(16)));

// The element's matrix operands, specialised beside each kernel: x8, eight elements; Weights, those of eight keys
// (set_pair(i, x, y) for an even i); product(a, b, c) and weighted(a, weights, c), kProducts of it, 32 x 32 += 32 x 16 times
// 16 x 32.
template <typename E>
struct TurnsOperand;

template <int D>
constexpr int turns_stage_bytes() {  // K or V
  return (int)kTurnsKeys * D * 2;
}
template <int D, bool SPLIT>
constexpr int turns_lds_bytes() {  // SPLIT: [group][K 0 | K 1 | V 0 | V 1], else [K 0 | K 1 | K 2 | V 0 | V 1 | V 2]
  return (SPLIT ? 8 : 6) * turns_stage_bytes<D>();
}
template <int D>
constexpr int turns_share_bytes() {  // SPLIT: what group 1 hands to group 0, in the stages' place
  return 4 * (D / 2 + 2) * 64 * 4;
}
template <bool SPLIT>
constexpr uint32_t turns_rows() {  // query rows of a workgroup
  return SPLIT ? 128 : 256;
}

// What each of WAVES waves copies of a stage of K or V: COUNT times KEYS rows.
template <int D, int WAVES, bool VALUES>
struct TurnsCopy {
  static constexpr int PIECES = D / 8, KEYS = 64 / PIECES, COUNT = (int)kTurnsKeys / KEYS / WAVES;
  static_assert(COUNT == 1 || COUNT == 2 || COUNT == 4, "copies");
  static __device__ __forceinline__ uint32_t row(uint32_t thread, int c) {
    return ((thread >> 6) % WAVES * COUNT + c) * KEYS + (thread & 63) / PIECES;
  }
  // where in its row the piece is that this lane leaves at its place
  static __device__ __forceinline__ uint32_t piece_bytes(uint32_t thread, int c) {
    return ((thread % PIECES) ^ ((VALUES ? 2 : 1) * row(thread, c) & (PIECES - 1))) * 16;
  }
  static __device__ __forceinline__ uint32_t target(uint32_t stage, uint32_t wave, int c) {
    return stage + (wave % WAVES * COUNT + c) * 1024;
  }
  // Where a lane reads for each copy of a stage whose rows are one stride behind each other; the instruction's own offset
  // moves both ends, so that all copies share an address and a target.
  uint32_t offset[COUNT], wave;
  __device__ __forceinline__ TurnsCopy(uint32_t stride_bytes, uint32_t thread)
      : wave((uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6))) {
#pragma unroll
    for (int c = 0; c < COUNT; ++c) offset[c] = row(thread, c) * stride_bytes + piece_bytes(thread, c) - c * 1024;
  }
  // the stage from `first` on, the same for the whole wave
  __device__ __forceinline__ void whole(const void *first, uint32_t stage) const {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (COUNT == 4)
      asm volatile("s_mov_b32 m0, %5\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %4\n\t"
                   "global_load_lds_dwordx4 %1, %4 offset:1024\n\tglobal_load_lds_dwordx4 %2, %4 offset:2048\n\t"
                   "global_load_lds_dwordx4 %3, %4 offset:3072"
                   : : "v"(offset[0]), "v"(offset[1]), "v"(offset[2]), "v"(offset[3]), "s"(first), "s"(target(stage, wave, 0))
                   : "memory");
    else if constexpr (COUNT == 2)
      asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %2\n\t"
                   "global_load_lds_dwordx4 %1, %2 offset:1024"
                   : : "v"(offset[0]), "v"(offset[1]), "s"(first), "s"(target(stage, wave, 0)) : "memory");
    else
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                   : : "v"(offset[0]), "s"(first), "s"(target(stage, wave, 0)) : "memory");
#endif
  }
  // row r of the stage at from(r)
  template <typename From>
  __device__ __forceinline__ void rows(const From &from, uint32_t stage) const {
#if defined(__HIP_DEVICE_COMPILE__)
    uint32_t thread = threadIdx.x;
    asm volatile("" : "+v"(thread));  // (these stages are few: nothing of theirs is kept in registers for all of them)
#pragma unroll
    for (int c = 0; c < COUNT; ++c) {
      const char *source = reinterpret_cast<const char *>(from(row(thread, c))) + piece_bytes(thread, c);
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                   : : "v"(source), "s"(target(stage, wave, c)) : "memory");
    }
#endif
  }
};

__device__ __forceinline__ void both_halves(float v, float &low, float &high) {
  const auto swapped = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v),
                                                        false, false);
  low = __builtin_bit_cast(float, (uint32_t)swapped[0]), high = __builtin_bit_cast(float, (uint32_t)swapped[1]);
}

// The keys low .. high of a lane's query row, of the wave's rows the first and last of both, and whether any of the rows exist (the
// same for the wave).
struct TurnsBounds {
  uint32_t low, high, low_first, low_last, high_first, high_last;
  bool rows;
};

// How a score s becomes an exponent to base two: s * inner (inner > 0); cap tanh, by inner = 2 scale / softcap * log2 e and
// cap = softcap * log2 e; the same under a cap that bounds it, where `top` is constant.
enum class TurnsScores { kPlain, kCapped, kFixed };

// out, top and total of this lane's row (total: of this lane's keys; both halves together are the row's) over the keys
// begin .. begin + 64 stages - 1 as far as `bounds` lets them be seen; on the way in they hold what the row starts with
// (SPLIT: in group 0).  False: another wave has the row (SPLIT, group 1).  copy_k / copy_v(key, stage): this wave's part of
// the 64 rows from `key` on into a stage in LDS.
template <typename E, int D, bool SPLIT, TurnsScores SCORES, typename CopyK, typename CopyV>
__device__ __forceinline__ bool attention_turns(unsigned char *lds, const typename TurnsOperand<E>::x8 (&q)[D / 16],
                                                const TurnsBounds &bounds, uint32_t begin, uint32_t stages, float inner,
                                                float cap, float &top, float &total, f32x16 (&out)[D / 32],
                                                const CopyK &copy_k, const CopyV &copy_v) {
  typedef TurnsOperand<E> Operand;
  typedef typename Operand::x8 x8;
  constexpr int KSTEPS = D / 16, JJ = D / 32, ROW = D * 2, PIECES = D / 8, STAGE = turns_stage_bytes<D>();
  constexpr int kCopies = 2 * TurnsCopy<D, SPLIT ? 4 : 8, false>::COUNT;
  constexpr uint32_t RING = SPLIT ? 2 : 3, EVERY = SPLIT ? 2 : 1;  // stages in LDS; every which stage is this group's
  const uint32_t lane = threadIdx.x & 63, row_lane = lane & 31, half = lane >> 5;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), group = wave >> 2;
  unsigned char *own = lds + (SPLIT ? group * 4 * STAGE : 0);
  const uint32_t own_address = (uint32_t)(size_t)(__attribute__((address_space(3))) unsigned char *)own;
  const uint32_t start = begin + (SPLIT ? group * kTurnsKeys : 0);
  const uint32_t steps = (stages + EVERY - 1) / EVERY, here = SPLIT ? (stages + 1 - group) / 2 : stages;  // here: this group's
  const auto first_key = [&](uint32_t step) { return start + step * (EVERY * kTurnsKeys); };
  const auto k_place = [&](uint32_t step) { return step % RING * STAGE; };
  const auto v_place = [&](uint32_t step) { return (RING + step % RING) * STAGE; };

  // a lane's places in the stages: K row row_lane (pieces ks * 2 + half, XOR-ed), and what it names in a transposing read
  const uint32_t k_lane = row_lane * ROW + ((half ^ (row_lane & (PIECES - 1))) * 16);
  uint32_t v_lane[JJ];
  {
    const uint32_t part = lane >> 4, p = lane & 15, key = (part >> 1) * 4 + (p >> 2), chunk = (part & 1) * 4 + (p & 3);
#pragma unroll
    for (int jj = 0; jj < JJ; ++jj)
      v_lane[jj] = key * ROW + (((jj * 4 + (chunk >> 1)) ^ ((2 * key) & (PIECES - 1))) * 16) + (chunk & 1) * 8;
  }

  if (here > 0) copy_k(first_key(0), own_address + k_place(0)), copy_v(first_key(0), own_address + v_place(0));
  if (here > 1) copy_k(first_key(1), own_address + k_place(1));
  copies_landed<0>();
  meet();
  if (group == 1) meet();

  // in the other steps the wave only copies and waits
  const auto [first, last] = turns_steps(bounds.rows, bounds.low_first, bounds.high_last, start, EVERY, here);

  f32x16 score[2];
  typename Operand::Weights weights[4];
  const auto scores = [&](uint32_t step) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) score[t][r] = 0.0f;
    const unsigned char *rows = own + k_place(step);
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks)
#pragma unroll
      for (int t = 0; t < 2; ++t)
        score[t] = Operand::product(*reinterpret_cast<const x8 *>(rows + t * 32 * ROW + (k_lane ^ (ks * 32))), q[ks], score[t]);
  };
  const auto values = [&](uint32_t step) __attribute__((always_inline)) {
    typedef short s4_t __attribute__((ext_vector_type(4)));
    typedef s4_t __attribute__((address_space(3))) * lds_chunk_t;
    // A weight of zero times an infinite value is NaN: 32 keys that no row of the wave sees take the values of the other 32.
    const uint32_t key = first_key(step);
    const unsigned char *stage = own + v_place(step);
    const unsigned char *rows[2] = {stage + (bounds.low_first > key + 31 ? 32 * ROW : 0), stage + (bounds.high_last < key + 32 ? 0 : 32 * ROW)};
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int jj = 0; jj < JJ; ++jj) {
        const unsigned char *from = rows[s / 2] + v_lane[jj] + s % 2 * 16 * ROW;
        const s4_t low = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_chunk_t)from);
        const s4_t high = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_chunk_t)(from + 8 * ROW));
        const x8 operand = __builtin_bit_cast(x8, __builtin_shufflevector(low, high, 0, 1, 2, 3, 4, 5, 6, 7));
        out[jj] = Operand::weighted(operand, weights[s], out[jj]);
      }
  };
  // a step's weights begin and end with these
  const auto begin_weights = [&](uint32_t step) __attribute__((always_inline)) {
    if (!SPLIT && group == 1) copies_landed<0>();
    meet();
    if (step + 1 < here) copy_v(first_key(step + 1), own_address + v_place(step + 1));
    if (step + 2 < here) copy_k(first_key(step + 2), own_address + k_place(step + 2));
  };
  const auto end_weights = [&](uint32_t step) __attribute__((always_inline)) {
    if (SPLIT || group == 0) {  // all but the copies that this step has asked for
      if (step + 2 < here) copies_landed<kCopies>();
      else copies_landed<0>();
    }
    meet();
  };
  const auto idle = [&](uint32_t step) __attribute__((always_inline)) {
    begin_weights(step);
    end_weights(step);
  };
  if (first >= last) {
    for (uint32_t step = 0; step < steps; ++step) idle(step);
  } else {
    for (uint32_t step = 0; step < first; ++step) idle(step);
    scores(first);
    for (uint32_t step = first; step < last; ++step) {
      begin_weights(step);
      const uint32_t key = first_key(step);
      const bool whole = key >= bounds.low_last && key + kTurnsKeys - 1 <= bounds.high_first;
      const auto mask = [&](float hidden) {
        const uint32_t from = bounds.low - key - half * 4, count = bounds.high - bounds.low;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            score[t][r] = (uint32_t)(t * 32 + (r >> 2) * 8 + (r & 3)) - from <= count ? score[t][r] : hidden;
      };
      if constexpr (SCORES != TurnsScores::kPlain) {
        const float high = SCORES == TurnsScores::kFixed ? cap - top : cap;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const float tail = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(score[t][r] * inner));
            score[t][r] = fmaf(-2.0f * cap, tail, high);
            if (SCORES == TurnsScores::kFixed) score[t][r] = __builtin_amdgcn_exp2f(score[t][r]);
          }
      }
      if (!whole) mask(SCORES == TurnsScores::kFixed ? 0.0f : -INFINITY);
      if constexpr (SCORES != TurnsScores::kFixed) {
        float best = score[0][0];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r) best = fmaxf(best, score[t][r]);
        float low, high;
        both_halves(best, low, high);
        best = fmaxf(low, high) * (SCORES == TurnsScores::kPlain ? inner : 1.0f);
        const bool above = best > top;
        if (__builtin_amdgcn_ballot_w64(above) != 0) {
          const float higher = above ? best : top;
          const float alpha = __builtin_amdgcn_exp2f(top - higher);
          top = higher;
          total *= alpha;
#pragma unroll
          for (int jj = 0; jj < JJ; ++jj)
#pragma unroll
            for (int r = 0; r < 16; ++r) out[jj][r] *= alpha;
        }
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            score[t][r] = __builtin_amdgcn_exp2f(SCORES == TurnsScores::kPlain ? fmaf(score[t][r], inner, -top) : score[t][r] - top);
      }
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
          total += score[t][r];
          total += score[t][r + 1];
          weights[t * 2 + (r >> 3)].set_pair(r & 7, score[t][r], score[t][r + 1]);
        }
      asm volatile("" : "+v"(total));  // here, and not with all weights in registers behind the products
      end_weights(step);
      if (group == 1) __builtin_amdgcn_s_setprio(1);  // against the older wave's softmax
      scores(step + 1);  // (behind the last step they are of whatever is there, and nothing reads them)
      values(step);
      // operands come from LDS four ahead of their products
      constexpr int kProduct = 0x8, kRead = 0x100, kAhead = 4, kScores = 2 * KSTEPS, kValues = 4 * JJ;
      __builtin_amdgcn_sched_group_barrier(kRead, kAhead, 0);
#pragma unroll
      for (int i = 0; i < kScores - kAhead; ++i) {
        __builtin_amdgcn_sched_group_barrier(kProduct, 1, 0);
        __builtin_amdgcn_sched_group_barrier(kRead, 1, 0);
      }
#pragma unroll
      for (int i = 0; i < kAhead; ++i) {
        __builtin_amdgcn_sched_group_barrier(kProduct, 1, 0);
        __builtin_amdgcn_sched_group_barrier(kRead, 2, 0);
      }
#pragma unroll
      for (int i = 0; i < kValues - kAhead; ++i) {
        __builtin_amdgcn_sched_group_barrier(kProduct, Operand::kProducts, 0);
        __builtin_amdgcn_sched_group_barrier(kRead, 2, 0);
      }
      __builtin_amdgcn_sched_group_barrier(kProduct, kAhead * Operand::kProducts, 0);
      if (group == 1) __builtin_amdgcn_s_setprio(0);
    }
    for (uint32_t step = last; step < steps; ++step) idle(step);
  }
  if (group == 0) meet();

  meet();
  if constexpr (!SPLIT) return true;
  // Group 1's share in the place of the stages, register by register with the lanes side by side: both waves of a row hold
  // the same (row, component) in the same lane and register.
  float *share = reinterpret_cast<float *>(lds) + (wave & 3) * (JJ * 16 + 2) * 64 + lane;
  static_assert(turns_share_bytes<D>() <= turns_lds_bytes<D, true>(), "the shares fit the stages");
  if (group == 1) {
    share[0] = top, share[64] = total;
#pragma unroll
    for (int jj = 0; jj < JJ; ++jj)
#pragma unroll
      for (int r = 0; r < 16; ++r) share[(2 + jj * 16 + r) * 64] = out[jj][r];
    lds_read();
  }
  meet();
  if (group == 1) return false;
  const float its_top = share[0], best = fmaxf(top, its_top);
  const float mine = __builtin_amdgcn_exp2f(top - best), its = __builtin_amdgcn_exp2f(its_top - best);
  total = total * mine + share[64] * its;
#pragma unroll
  for (int jj = 0; jj < JJ; ++jj)
#pragma unroll
    for (int r = 0; r < 16; ++r) out[jj][r] = out[jj][r] * mine + share[(2 + jj * 16 + r) * 64] * its;
  return true;
}

// A wave's 32 rows as halves of eight bytes a lane and place, to rows of `stride` elements from `target` on, `count` of them:
// through LDS (the wave's own 32 * (D * 2 + 16) bytes), so that sixteen lanes store a row.
template <int D, typename Pack>
__device__ __forceinline__ void store_rows(unsigned char *lds, void *target, size_t stride_bytes, uint32_t count, const Pack &pack) {
  constexpr int ROW = D * 2 + 16, PIECES = D / 8, AT_ONCE = 64 / PIECES;
  typedef uint32_t piece_t __attribute__((ext_vector_type(4), aligned(8)));  // (rows may start at any eight bytes)
  const uint32_t lane = threadIdx.x & 63, row_lane = lane & 31, half = lane >> 5;
#pragma unroll
  for (int jj = 0; jj < D / 32; ++jj)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<uint2 *>(lds + row_lane * ROW + (32 * jj + g * 8 + half * 4) * 2) = pack(jj, 4 * g);
  lds_read();
#pragma unroll
  for (int i = 0; i < 32 / AT_ONCE; ++i) {
    const uint32_t row = i * AT_ONCE + lane / PIECES, piece = lane % PIECES * 16;
    const piece_t whole = *reinterpret_cast<const piece_t *>(lds + row * ROW + piece);
    if (row < count) *reinterpret_cast<piece_t *>(static_cast<char *>(target) + row * stride_bytes + piece) = whole;
  }
}
template <int D>
constexpr int store_rows_bytes() {
  return 32 * (D * 2 + 16);
}

}  // namespace llmopt
