// How many workgroups a compute unit the gated delta rule's chunk kernel runs: a rule on sizes alone, without HIP, so that a
// host test can ask it.
#pragma once

#include <stdint.h>

namespace llmopt {

// Heads of up to 128: a third workgroup a compute unit costs the registers' last ten a trip to scratch, and is the better one
// where it saves a round of workgroups: 3001 tokens of 16 heads, 752 workgroups, one round for two, 71 us for 98 (in float32
// the whole rule 264 for 332), but not of 8 heads, 376 workgroups, 48 for 45.5, nor 4096 tokens of 16 heads, 1024 workgroups
// and two rounds either way (the whole rule of value heads of 64 245 us for 224).  LDS (53 KB) holds three.  Heads of 64 fit
// anyway, wider ones take all registers.
inline bool three_delta_workgroups(uint64_t workgroups, uint32_t cus) {
  auto rounds = [&](uint64_t each) { return (workgroups + each * cus - 1) / (each * cus); };
  return rounds(3) < rounds(2);
}

}  // namespace llmopt
