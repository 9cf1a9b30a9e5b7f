// Which tile a bfloat16 product takes: a rule on sizes alone (and the number of compute units), without HIP, so that a host
// test can ask it.
#pragma once

#include <stdint.h>

namespace llmopt {

enum class DenseTile { k256x256, k128x128, k192x128, k128x192, k192x128Eight, k128x128Eight, k64x128Eight, k64x64, k32x64, k64x128 };

// Tiles in that order, and what a round of them takes on 256 CUs at K = 2048 (us, weights from HBM; a round's time goes with
// K): with one workgroup on a CU, and with two where the tile's ring leaves room for them.  The eight-wave tiles keep two
// stages of copies under way instead of one, which covers the trip to HBM when a CU has no second workgroup to fill the wait.
struct TileRound {
  uint32_t rows, columns;
  float one, two;  // two == 0: the ring takes the CU
};
constexpr TileRound kTileRounds[] = {
    {256, 256, 53.0f, 0.0f},  // 8 waves, 2 stages
    {128, 128, 31.0f, 38.0f}, // 4 waves, 2 stages
    {192, 128, 34.0f, 52.0f}, // 4 waves, 2 stages
    {128, 192, 35.0f, 55.0f}, // 4 waves, 2 stages
    {192, 128, 29.0f, 0.0f},  // 8 waves, 3 stages
    {128, 128, 23.0f, 0.0f},  // 8 waves, 3 stages
    {64, 128, 15.3f, 0.0f},   // 8 waves, 4 stages
    {64, 64, 11.2f, 17.0f},   // 4 waves, 4 stages
    {32, 64, 8.5f, 13.7f},    // 4 waves, 6 stages
};

// The tile with the least time by these (columns: a gated pair's both matrices).  Measured, us (m x n x k), before (the
// largest tile that gives every CU work) and now: 2048 x 2048 x 4096 58 / 47, 2048 x 2048 x 8192 97 / 86, 2048 x 8576 x 2048
// 94 / 80, 2048 x 6144 x 2048 69 / 56, 3001 x 2048 x 4096 67 / 63, 1024 x 2048 x 4096 34 / 31, 512 x 6144 x 2048 28 / 23;
// 3001 x 9504 x 2048 118, 512 x 2048 x 4096 22, 64 x 4384 x 1024 7.0 as before.  Over 720 sizes (K 64 to 8192, 512 to 16384
// columns, 2 to 3001 rows) it is 4% faster than that rule on average and 1% off the best tile.  It is furthest off with a few
// tiles of 64 x 64 more than CUs, which it counts as two on every CU: 700 x 1500 x 8192 51 for 42, 1500 x 1024 x 4096 29
// for 27 (1024 x 1500 x 4096 is the other way round, 29 for 33).
// With a short K the start and the end of a workgroup decide, not its steps: where the estimate takes 128 x 128 tiles of eight
// waves, twice as many of 64 x 128 and four waves, several on a CU, are over sooner (700 x 4096 x 128 7.6 / 7.0, 1500 x 2048 x
// 128 7.25 / 7.0, 3001 x 1024 x 256 8.45 / 8.1, 700 x 4096 x 256 8.6 / 7.95; at K = 64 the same either way, at 512 11.2 / 12.2).
inline DenseTile dense_tile(uint32_t m, uint64_t columns, uint32_t k, uint32_t cus) {
  int best = 0;
  float least = 3.4e38f;
  for (int i = 0; i < (int)(sizeof(kTileRounds) / sizeof(kTileRounds[0])); ++i) {
    const TileRound &t = kTileRounds[i];
    const uint64_t tiles = ((m + t.rows - 1) / t.rows) * ((columns + t.columns - 1) / t.columns);
    const uint64_t slots = t.two > 0.0f ? 2ull * cus : cus, rest = tiles % slots;
    const float full = t.two > 0.0f ? t.two : t.one;
    const float time = (float)(tiles / slots) * full + (rest == 0 ? 0.0f : rest <= cus ? t.one : t.two);
    if (time < least) least = time, best = i;
  }
  const DenseTile tile = (DenseTile)best;
  return tile == DenseTile::k128x128Eight && k > 64 && k <= 256 ? DenseTile::k64x128 : tile;
}

}  // namespace llmopt
