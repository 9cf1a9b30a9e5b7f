// Which dense attention launches take two groups of waves in turns, and which of the key-splitting ones eight waves a slab:
// rules on sizes alone, without HIP, so that a host test can ask them.
#pragma once

#include <stdint.h>

namespace llmopt {

// The key / value head of a query head; the query heads are a multiple of them.  (head * kv_heads / heads is one division fewer
// and wraps from 2^32 on: 131072 heads over 65536.)
constexpr uint32_t kv_head_of(uint32_t head, uint32_t heads, uint32_t kv_heads) {
  return kv_heads < heads ? head / (heads / kv_heads) : head;
}

// The waves of a workgroup share 32 query rows and a stage of 32 keys each.  One workgroup per CU that walks several stages:
// eight waves and 256-key stages (128 KB) halve the walk again (us, query rows / keys they see / heads, eight / four waves:
// 700 / 700 / 9 8.3 / 8.5, 900 / 900 / 9 9.6 / 10.4, 64 / 2000 / 9 12.5 / 14.2, 400 / 4000 / 9 19.8 / 24.0).  Walks of a few
// stages are as short either way (512 / 512 / 9 7.2 / 7.4, 300 rows that see 300 of 900 keys 7.0 / 6.7, 400 of 4000 7.4 / 7.5, 32
// that see 32 of 4096 6.8 / 6.8), and where two workgroups would share a CU that room is worth more (700 / 700 / 32 16.0 / 12.1,
// 2048 / 2048 / 9 21.0 / 17.2).
// A few slabs more than CUs are a second round, which is short under a causal limit once the walk is long (32 slabs of 9 heads
// over 1000 keys 9.4 / 10.0; 18 of 16 heads over 560 8.7 / 8.1) and as long as the first without one (18 of 16 heads over
// 560 12.0 / 9.5).  With a mask the map of stages counts in 128 keys.
inline bool eight_wave_slabs(uint32_t head_dim, bool masked, bool causal, uint32_t query_length, uint32_t key_length,
                             uint32_t past_length, uint64_t slabs, uint32_t cus) {
  const uint64_t last = (uint64_t)past_length + query_length;  // keys that the last row sees under a causal limit
  const uint64_t walk = causal && last < key_length ? last : key_length;
  const uint64_t room = causal && walk > 640 ? (uint64_t)cus * 9 / 8 : cus;
  return head_dim == 64 && !masked && key_length > 512 && walk > 256 && slabs <= room;
}

// Forms that keep a value row's place behind its stage's first one in 32 bits, for up to 63 rows of halves.
constexpr bool short_value_rows(uint64_t value_row_halfs) { return value_row_halfs < (1u << 25); }

// Workgroups of 512 threads in a grid, which has fewer than 2^32 threads.  Workgroups of 256 go on to twice as many.
constexpr bool turns_grid(uint64_t workgroups) { return workgroups * 512 < (1ull << 32); }

enum class TurnsForm { kNone, kSplit, kRows };

// Without a mask, from 256 keys on (below that the groups have a stage or two each); workgroups: of 128 rows.
// kSplit, 128 rows whose keys the groups share, against the key-splitting slabs of 32 rows, of which there is a workgroup a CU at
// most once there are as many of 128 rows as CUs.  Heads of 128 from half of the CUs on (us, heads x rows: 32 x 700 16.5 / 21.4,
// 16 x 1200 21.5 / 25.9, 16 x 1900 32 / 47, 8 x 3000 42 / 51; at half of them 32 x 500 13.8 / 14.7, 4 x 4096 54.1 / 53.6, 16 x 900 18.5 /
// 16.9; 16 x 700 15.5 / 12.3, 32 x 300 10.8 / 9.9), heads of 64, two slabs of which fit a CU, not before (32 x 1000 15.2 / 23.2,
// 9 x 3600 39 / 73; 32 x 800 12.8 / 12.8, 9 x 3500 37.2 / 35.5, 16 x 1900 23.7 / 21.3, 9 x 2048 24.5 / 16.2).
// kRows, 256 rows and their own group each, half the copies and no sums to hand over, once the longer workgroups still come to
// more than a round and a half (32 heads of 128: 4096 rows 162 / 167, 3500 126 / 131, 3000 102 / 100, 2048 62 / 48), and
// only where rows fill them.
// Beyond two workgroups a CU there is more to do than the longest one, and workgroups of four waves that share a CU freely hide
// their starts and ends behind each other; both groups in turns walk to the end together.  How long a workgroup walks on average
// decides: on short walks turns lose what they gain on long ones, and heads that share their keys gain most (us, turns / four waves:
// 16 heads of 128, 30 sequences of 520 tokens 139 / 99, 7 of 668 40.5 / 34.4; 128 rows of 600 keys, 75 x 32 over 8 heads 251 / 183, 44 x
// 16 heads 69 / 63, 22 x 32 over 8 55 / 58, and of 1000 keys, 75 x 32 over 8 275 / 278; 9 over 3 heads of 64, 20 sequences of 520 tokens
// 34 / 27, 13 of 668 28.3 / 25.3, 13 of 668 after 332 others 41 / 43.5, 128 rows of 600 keys, 78 sequences, 38.8 / 38).
// kRows has fewer and longer workgroups (16 heads of 128: 17 sequences of 1030 tokens 150 / 150, 9 of 2048 206 / 230).
// Up to 32 rows a head leave three of four waves of each group idle, still less than what slabs of 32 rows took whose waves met at
// every stage (130 over 13 heads of 128, 16 rows: 1000 keys 18.2 / 22, 4000 keys 49.5 / 66.7); their own tiles take 16.5 and 44.4.
inline TurnsForm turns_form(uint32_t head_dim, bool masked, bool causal, uint32_t query_length, uint32_t key_length,
                            uint32_t past_length, uint64_t workgroups, uint64_t value_row_halfs, uint32_t cus) {
  if (!short_value_rows(value_row_halfs) || !turns_grid(workgroups)) return TurnsForm::kNone;
  if (masked || (head_dim != 64 && head_dim != 128) || key_length < 256) return TurnsForm::kNone;
  const uint64_t seen = (uint64_t)past_length + query_length / 2;  // by a row in the middle
  const uint64_t walk = causal && seen < key_length ? seen : key_length;
  if (workgroups > 3 * (uint64_t)cus) {
    if (query_length >= 1024 && key_length >= 512) return TurnsForm::kRows;
    return walk >= 900 ? TurnsForm::kSplit : TurnsForm::kNone;
  }
  if (workgroups > 2 * (uint64_t)cus) return walk >= (head_dim == 64 ? 500 : 700) ? TurnsForm::kSplit : TurnsForm::kNone;
  return (head_dim == 64 ? workgroups >= cus : 2 * workgroups > cus) ? TurnsForm::kSplit : TurnsForm::kNone;
}

// The same over a portion of a prompt in bfloat16, 128 rows and their keys shared.  A workgroup starts and ends in some 8 us of
// which nothing overlaps, so that it pays for long walks; how long is known from the rows and the span alone (earlier portions'
// keys only make it longer).  us, heads x rows of span, turns / 16-row tiles: heads of 128 16 x 3001 of 2048 75 / 96, 32 x 3001 of
// 1024 102 / 118, 16 x 700 28 / 31, 16 x 500 25.1 / 25.8, 32 x 1500 of 512 54.5 / 53.9; of 64 16 x 3001 of 2048 51 / 60, 16 x 1500
// 33 / 37, 16 x 3001 of 1024 46.6 / 45.6.  A cap's two more exponentials a score hide better behind four waves a SIMD: heads of
// 128 32 x 2048 74 / 90, 32 x 3001 of 1024 70 / 80, 32 x 1000 34 / 34, 32 x 2000 of 512 40 / 35; of 64 16 x 2048 41 / 40.
inline bool chunk_turns(uint32_t dim, bool capped, uint32_t m, uint32_t span, uint32_t heads) {
  if (!turns_grid((uint64_t)heads * ((m + 127) / 128))) return false;
  const uint32_t walk = span != 0 && span < m ? span : m;
  if (dim == 128) return walk > (capped ? 1000 : 512);
  return dim == 64 && !capped && walk > 1024;
}

// The head that workgroup `rank` of a slab takes.  Workgroups go to the eight XCDs in turn: the heads of a key head follow each other
// eight apart, on one XCD's L2 when the key heads come in whole eights, and soon, while its keys are still there (3000 heads of 128
// over 750, 128 rows of 1500 keys: kv_heads apart 533 us, so 416).
constexpr uint32_t turns_head(uint32_t rank, uint32_t heads, uint32_t kv_heads) {
  const uint32_t per = heads / kv_heads, first = rank / (8 * per) * 8, left = kv_heads - first, width = left < 8 ? left : 8;
  const uint32_t at = rank - first * per;
  return (first + at % width) * per + at / width;
}

constexpr uint32_t kTurnsKeys = 64;  // of a stage

// The steps first .. last - 1 (none if first >= last) of `here`, one for the 64 keys behind start + step * every * 64, that hold keys
// which a wave's rows see: its first row from low_first on, its last one up to high_last.  A wave whose rows all lie past the end
// sees none, it only copies and waits: 700 rows leave half of every head's last and longest slab to such waves.
struct TurnsSteps {
  uint32_t first, last;
};
constexpr TurnsSteps turns_steps(bool any_rows, uint32_t low_first, uint32_t high_last, uint32_t start, uint32_t every, uint32_t here) {
  const uint32_t apart = every * kTurnsKeys;
  const uint32_t first = low_first > start ? (low_first - start + (every - 1) * kTurnsKeys) / apart : 0;
  const uint32_t end = high_last < start || !any_rows ? 0 : (high_last - start) / apart + 1;
  return {first, end < here ? end : here};
}

}  // namespace llmopt
