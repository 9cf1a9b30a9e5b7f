// Which of its tiles a prompt's W4A16 product takes: a rule on sizes (and the number of compute units) without HIP, so that a
// host test can ask it.
#pragma once

#include <stdint.h>

namespace llmopt {

// (deep: four activation stages)
enum class W4GemmTile { k128x128, k128x128Deep, k256x128, k128x256, k256x256 };

// The 256 x 256 tiles hold offsets from a tile's first row in 32 bits: 256 rows of K halves.
constexpr uint32_t kW4OffsetK = 1u << 22;

// Tall (256 x 128) or wide (128 x 256) tiles, whichever pads less; the tall one when they tie (its waves read 16 operand vectors
// from LDS per 16 MFMAs, the wide one's 20: 76.5 against 80 us at 512 x 14336, 81.7 against 86.3 at 2048 x 4096).  Also when a
// few CUs stay without a tile: 224 such tiles beat 448 of 128 x 128, two on most CUs.
// 256 x 256 once even the better of those would begin a second round: us, 256 x 128 or 128 x 256 / 256 x 256: 2048 x 2048 x 6144
// 82 / 63, 1024 x 4096 x 14336 154 / 118, 1430 x 576 x 5632 30.5 / 22.9; where they are one round 1134 x 2112 x 6720 45 / 55, 541 x
// 576 x 11840 20 / 23.
// 128 x 128 tiles have steps shorter than a trip to memory.  With two stages they fit a CU twice, which covers the loads; when
// there is at most one tile per CU anyway, four activation stages do (measured 58 -> 49 us at 512 x 4096 x 4096, and nothing for
// the 128 x 256 tiles, which stay with two).
inline W4GemmTile w4_gemm_tile(uint32_t m, uint32_t n, uint32_t k, uint32_t cus) {
  const uint64_t tall = (uint64_t)((m + 255) / 256) * ((n + 127) / 128), wide = (uint64_t)((m + 127) / 128) * ((n + 255) / 256);
  const uint64_t fewer = tall < wide ? tall : wide, small = (uint64_t)((m + 127) / 128) * ((n + 127) / 128);
  if (fewer > cus && k <= kW4OffsetK) return W4GemmTile::k256x256;
  if (fewer * 8 >= (uint64_t)cus * 7) return tall <= wide ? W4GemmTile::k256x128 : W4GemmTile::k128x256;
  return small <= cus ? W4GemmTile::k128x128Deep : W4GemmTile::k128x128;
}

// A gated pair, by output columns (128 x 128 outputs: both matrices' 128 columns; 256 x 256: 128 outputs a row).  256 x 256 once the
// deep 128 x 128 tiles would begin a second round.
inline W4GemmTile w4_gemm_pair_tile(uint32_t m, uint32_t n, uint32_t k, uint32_t cus) {
  const uint64_t small = (uint64_t)((m + 127) / 128) * ((n + 127) / 128);
  return small > cus && k <= kW4OffsetK ? W4GemmTile::k256x256 : W4GemmTile::k128x128Deep;
}

}  // namespace llmopt
