// Which launches of one token's attention join their shares of the keys themselves (chunk_decode.h); a host test asks it too.
#pragma once

#include <stdint.h>

namespace llmopt {

// Whether the last workgroup of each key / value head joins its shares.  That saves a launch, and with one live share the
// arrival too, but one workgroup does for all the head's queries what the merge spreads over a workgroup each.  us a call,
// merge / join, query heads over key heads x width, at the ring's end and (first) with one live share:
//   16 over 4 x 64 (256 outputs a key head)    6.5 / 4.5;  2 shares 6.6 / 6.2, 16 9.7 / 6.7, 17 10.1 / 8.8, 64 22.8 / 15.2
//   32 over 8 x 128 (512)                      8.1 / 5.8;  2 shares 8.2 / 8.0, 16 11.2 / 9.7, 17 11.6 / 12.9, 64 27.3 / 25.2
//   64 over 4 x 64 (1024)                      7.2 / 5.3;  2 shares 7.4 / 8.5, 8 7.5 / 8.6, 16 10.6 / 12.9
constexpr uint32_t kJoinOutputs = 512, kJoinShares = 16, kJoinOutputsOfMore = 256, kJoinMostShares = 64;
// splits: the most shares that a token of the ring can have; counters: arrival counters at hand; lds_words: the least that a
// workgroup has (two words a share and head, one a head, and one).
inline bool joins(uint32_t splits, uint32_t heads, uint32_t kv_heads, uint32_t vdim, uint32_t counters, uint32_t lds_words) {
  const uint64_t per = heads / kv_heads;
  return kv_heads <= counters && splits > 1 && splits <= kJoinMostShares && per * vdim <= (splits <= kJoinShares ? kJoinOutputs : kJoinOutputsOfMore) &&
         per * (2 * splits + 1) + 1 <= lds_words;
}

}  // namespace llmopt
