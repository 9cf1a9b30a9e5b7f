// Which launch of the key-splitting dense attention takes eight waves a slab: a rule on sizes alone, without HIP, so that a
// host test can ask it.
#pragma once

#include <stdint.h>

namespace llmopt {

// The waves of a workgroup share 32 query rows and a stage of 32 keys each.  One workgroup per CU that walks several stages:
// eight waves and 256-key stages (128 KB) halve the walk again (us, query rows / keys they see / heads, eight / four waves:
// 700 / 700 / 9 10.2 / 11.5, 900 / 900 / 9 11.7 / 14.5, 64 / 2000 / 9 15.1 / 17.3, 400 / 4000 / 9 29.8 / 40.5).  Walks of a few
// stages are as short either way (512 / 512 / 9 8.4 / 8.3, 300 rows that see 300 of 900 keys 10.6 / 10.6; 400 of 4000 11.0 /
// 11.7) or shorter with four (32 rows that see 32 of 4096 keys 8.7 / 8.0, 100 that see 100 of 520 9.0 / 8.5), and where two
// workgroups would share a CU that room is worth more (700 / 700 / 32 20.6 / 14.0, 2048 / 2048 / 9 26.7 / 20.0).
// A few slabs more than CUs are a second round, which is short under a causal limit once the walk is long (32 slabs of 9 heads
// over 1000 keys 15.0 / 17.5; 18 of 16 heads over 560 14.2 / 13.5) and as long as the first without one (18 of 16 heads over
// 560 20.2 / 15.0).  With a mask the map of stages counts in 128 keys.
inline bool eight_wave_slabs(uint32_t head_dim, bool masked, bool causal, uint32_t query_length, uint32_t key_length,
                             uint32_t past_length, uint64_t slabs, uint32_t cus) {
  const uint64_t last = (uint64_t)past_length + query_length;  // keys that the last row sees under a causal limit
  const uint64_t walk = causal && last < key_length ? last : key_length;
  const uint64_t room = causal && walk > 640 ? (uint64_t)cus * 9 / 8 : cus;
  return head_dim == 64 && !masked && key_length > 512 && walk > 256 && slabs <= room;
}

}  // namespace llmopt
