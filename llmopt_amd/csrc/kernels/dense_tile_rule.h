// Which tile a bfloat16 product takes: a rule on sizes alone (and the number of compute units), without HIP, so that a host
// test can ask it.
#pragma once

#include <stdint.h>

namespace llmopt {

// (the turns: two groups of four waves that take stages in turn)
enum class DenseTile {
  k256x256, k128x128, k192x128, k128x192, k192x128Eight, k128x128Eight, k64x128Eight, k64x64, k32x64, k64x128,
  kTurns192x128, kTurns128x128, kTurns128x192, kTurns256x128, kTurns128x64
};

// The first ten in that order, and an estimate of a launch on 256 CUs (us, K in 1024, weights from HBM).  `start` comes once, and a
// round of workgroups takes a constant, its start and its outputs, and a part that goes with K: with one workgroup on a CU,
// and with two where the tile's ring leaves room for them (`two_k` == 0: it takes the CU).  A last round on few CUs takes the
// share `few` of a whole one, which grows evenly to the whole.  The step from one workgroup on a CU to two comes to the share
// `pair` with the first CU that has two and is whole once the share `span` of the CUs have.  The eight-wave tiles keep two
// stages of copies under way instead of one, which covers the trip to HBM when a CU has no second workgroup to fill the wait.
struct TileTime {
  uint32_t rows, columns;
  float start, one, one_k, few, two, two_k, pair, span;
};
constexpr TileTime kTileTimes[] = {
    {256, 256, 0.01f, 14.10f, 24.56f, 1.00f, 0.00f, 0.00f, 0.00f, 0.00f},     // (see dense_tile)
    {128, 128, 0.00f, 7.54f, 20.73f, 0.47f, 8.85f, 15.57f, 0.02f, 0.65f},     // 4 waves, 2 stages
    {192, 128, 0.00f, 7.79f, 14.79f, 1.00f, 11.91f, 19.36f, 1.00f, 0.06f},    // 4 waves, 2 stages
    {128, 192, 5.82f, 1.85f, 15.16f, 1.00f, 7.30f, 21.46f, 0.99f, 0.17f},     // 4 waves, 2 stages
    {192, 128, 0.00f, 6.73f, 12.92f, 0.99f, 0.00f, 0.00f, 0.00f, 0.00f},      // 8 waves, 3 stages
    {128, 128, 0.01f, 5.78f, 9.27f, 0.92f, 0.00f, 0.00f, 0.00f, 0.00f},       // 8 waves, 3 stages
    {64, 128, 1.22f, 2.87f, 6.83f, 0.91f, 0.00f, 0.00f, 0.00f, 0.00f},        // 8 waves, 4 stages
    {64, 64, 0.98f, 2.42f, 4.09f, 1.00f, 2.29f, 9.08f, 0.00f, 0.22f},         // 4 waves, 4 stages
    {32, 64, 1.84f, 1.05f, 3.37f, 0.97f, 1.18f, 7.21f, 0.96f, 0.38f},         // 4 waves, 6 stages
    {64, 128, 0.07f, 4.40f, 8.62f, 0.78f, 4.57f, 12.70f, 0.81f, 0.13f},       // 4 waves, 3 stages
};

// The tile with the least time by these (columns: a gated pair's both matrices).  The constants are a fit to all ten tiles at
// 1900 sizes (8 to 3001 rows, 64 to 16384 columns, K 64 to 8192; 600 MB of weights in turn, so that none is in a cache), weighed
// by what a wrong choice costs: the choice is 0.5% off the best tile on average, and 7% faster than the largest tile that gives
// every CU work, which is more than 3% ahead at 29 of them.  An estimate of rounds that go with K alone was 0.8% off, and
// behind that tile by more than 3% at 72 (us, that tile / such an estimate: 384 x 2816 x 8192 41.0 / 52.0, 700 x 1500 x 8192 41.5
// / 50.4, 300 x 12288 x 512 12.4 / 13.4: these are back; 384 x 3072 x 8192, with 288 tiles of 64 x 64, 43.6 / 52.5 is not).
// The row of 256 x 256 tiles is that of all their waves in step.  With half of them a barrier behind, as they run now, a launch is
// 0.82 to 0.97 of it; from K = 1024 on dense_product_tile asks for their own times, below it this row is the line.  Own times on
// the scale of the others (1.64, 11.58, 21.16, 0.67) chose 0.1% faster tiles on average at 795 sizes and 3 to 10% slower ones at nine
// (2283 x 4608 x 448 17.9 / 18.7 us, 918 x 11008 x 192 12.3 / 13.4); this row a slower one than the other nine at none.
inline DenseTile dense_tile(uint32_t m, uint64_t columns, uint32_t k, uint32_t cus, float *estimate = nullptr) {
  int best = 0;
  float least = 3.4e38f;
  for (int i = 0; i < (int)(sizeof(kTileTimes) / sizeof(kTileTimes[0])); ++i) {
    const TileTime &t = kTileTimes[i];
    const bool pairs = t.two_k > 0.0f;
    const uint64_t tiles = ((m + t.rows - 1) / t.rows) * ((columns + t.columns - 1) / t.columns);
    const uint64_t slots = pairs ? 2ull * cus : cus, rest = tiles % slots;
    const float one = t.one + t.one_k * (float)k / 1024.0f, two = pairs ? t.two + t.two_k * (float)k / 1024.0f : one;
    const float share = (float)rest / (float)cus;  // of the CUs, in the last round
    float time = t.start + (float)(tiles / slots) * two;
    if (share > 1.0f) {
      const float more = share - 1.0f < t.span ? (share - 1.0f) / t.span : 1.0f;
      time += one + (two - one) * (t.pair + (1.0f - t.pair) * more);
    } else if (rest > 0) {
      time += one * (t.few + (1.0f - t.few) * share);
    }
    if (time < least) least = time, best = i;
  }
  if (estimate != nullptr) *estimate = least;
  return (DenseTile)best;
}

// The same estimate for the tiles whose waves multiply and read at different times, one workgroup on a CU: a fit at 1700 sizes
// (8 to 3001 rows, 64 to 16384 columns, K 64 to 8192, 640 MB of weights in turn).
struct StaggeredTime {
  DenseTile tile;
  uint32_t rows, columns;
  float start, one, one_k, few;
};
constexpr StaggeredTime kStaggeredTimes[] = {
    {DenseTile::k256x256, 256, 256, 2.83f, 7.36f, 20.88f, 0.66f},      // 8 waves, 2 stages, half of them behind
    {DenseTile::kTurns192x128, 192, 128, 2.04f, 5.54f, 10.32f, 0.73f}, // 2 x 4 waves, 3 stages
    {DenseTile::kTurns128x128, 128, 128, 1.75f, 4.03f, 7.81f, 0.78f},  // 2 x 4 waves, 5 stages
    {DenseTile::kTurns128x192, 128, 192, 3.31f, 4.26f, 10.58f, 0.72f}, // 2 x 4 waves, 3 stages
    {DenseTile::kTurns256x128, 256, 128, 1.98f, 7.19f, 11.84f, 0.69f}, // 2 x 4 waves, 3 stages
    {DenseTile::kTurns128x64, 128, 64, 1.88f, 2.42f, 5.50f, 0.76f},    // 2 x 4 waves, 5 stages
};
static_assert(kStaggeredTimes[0].tile == DenseTile::k256x256);

// `columns` of the whole product.  Rows of outputs that are no whole pieces of eight are stored value by value, which takes 256 x 256
// tiles 15 us a round more and the others less: without the 6 us of difference 897 x 11657 x 1024 took 44.7 us for 40.5, 1223 x
// 9265 x 1408 51.7 for 49.1.
inline float staggered_time(const StaggeredTime &t, uint64_t tiles, uint64_t columns, uint32_t k, uint32_t cus) {
  const uint64_t rest = tiles % cus;
  const float one = t.one + t.one_k * (float)k / 1024.0f, odd = t.tile == DenseTile::k256x256 && columns % 8 != 0 ? 6.0f : 0.0f;
  return t.start + (float)(tiles / cus) * one + (rest > 0 ? one * (t.few + (1.0f - t.few) * (float)rest / (float)cus) : 0.0f) +
         odd * (float)((tiles + cus - 1) / cus);
}

// The ten's estimates are a fit of their own and come out longer than launches behind each other, which the staggered ones' are of:
// 1.07 times at the median of 470 sizes beyond 25 us, where the two are compared.  This puts them on one scale.
constexpr float kInStepScale = 0.93f;

// Where the staggered tiles begin: in turns from 1280 (below, what the meeting of two groups' sums costs is not made up for: 0.99 of
// the ten's time on average, up to 1.16), 128 x 128 ones, which have the most sums to a product, from 1792: from 1280 on 0.98 of the
// eight waves in step, but more than 3% slower at 5 of 18 sizes (us, in step / in turns: 223 x 10624 x 1408 16.8 / 17.5, 751 x 5312 x
// 1408 17.3 / 18.1; the medians of three GPUs), from 1792 on 0.95 and 2 of 13, beyond 2560 0.93 and none of 16.
inline uint32_t staggered_from_k(DenseTile tile) {
  if (tile == DenseTile::k256x256) return 1024;
  return tile == DenseTile::kTurns128x128 ? 1792 : 1280;
}

// The tile a product runs on: one of the ten, or from K = 1024 on one of the staggered ones where its estimate is less: 0.96 of the
// ten's time on average from there on (us, ten / this: 2048 x 2048 x 8192 74 / 63, 2048 x 2048 x 2048 23.2 / 21.1, 3001 x 2048 x 8192
// 100 / 83, 2048 x 6144 x 2048 51.7 / 48.1, 700 x 2048 x 2048 15.6 / 14.0, 1008 x 1088 x 4288 26.2 / 25.0).
inline DenseTile dense_product_tile(uint32_t m, uint64_t columns, uint32_t k, uint32_t cus, float *estimate = nullptr) {
  float least = 0.0f;
  DenseTile best = dense_tile(m, columns, k, cus, &least);
  least *= kInStepScale;
  for (const StaggeredTime &t : kStaggeredTimes) {
    if (k < staggered_from_k(t.tile)) continue;
    const uint64_t tiles = ((m + t.rows - 1) / t.rows) * ((columns + t.columns - 1) / t.columns);
    const float time = staggered_time(t, tiles, columns, k, cus);
    if (time < least) least = time, best = t.tile;
  }
  if (estimate != nullptr) *estimate = least;
  return best;
}

// Products that 32 x 64 tiles suit best leave CUs without a tile, and each stage of a tile takes what its trip and its barrier
// take, 0.28 us a stage of 64 values whatever the rest.  They run on the smallest of these whose tiles come to one a CU at most,
// with groups of waves that take the stages in turn (eight groups of two waves, four of four).  us, one group on 32 x 64 tiles /
// 32 x 32 / 16 x 32, weights from HBM: 64 x 1024 x 4096 17.9 / 12.1 / 9.9, x 2048 10.1 / 6.3 / 5.3, x 1024 6.5 / 4.7 / 4.2, x 512
// 4.8 / 4.1 / 3.8, x 256 4.1 / 3.8 / 3.6, x 128 3.0 / 3.2 / 3.2: from K = 256.  Where 32 x 32 tiles are more than the CUs, 32 x 64 ones
// in four groups: 500 x 1024 x 4096 18.4 / 15.6, x 1024 6.8 / 5.9, x 512 5.0 / 5.0, 64 x 8192 x 1024 7.95 / 7.98: from K = 1024.
// A pair needs both matrices in a wave, which the smaller ones do not hold: 32 x 64 as well, beyond a quarter of the CUs from K = 2048
// (of single matrices 16 x 4096 x 1024 7.12 / 7.13, 16 x 8192 x 1024 7.39 / 7.56, x 2048 11.7 / 11.6).
enum class DenseParts { kNone, k16x32, k32x32, k32x64 };
inline DenseParts dense_parts(DenseTile tile, uint32_t m, uint64_t columns, uint32_t k, bool pair, uint32_t cus) {
  const auto tiles = [&](uint32_t rows, uint32_t wide) { return (uint64_t)((m + rows - 1) / rows) * ((columns + wide - 1) / wide); };
  if (tile != DenseTile::k32x64 || k < 256) return DenseParts::kNone;
  if (!pair && tiles(16, 32) <= cus) return DenseParts::k16x32;
  if (!pair && tiles(32, 32) <= cus) return DenseParts::k32x32;
  return k >= (pair && tiles(32, 64) > cus / 4 ? 2048 : 1024) && tiles(32, 64) <= cus ? DenseParts::k32x64 : DenseParts::kNone;
}

// A product in two launches: the first `columns` on whole rounds of 256 x 256 tiles, the rest on the tile that suits it (0: one
// launch).  A round of the 256 CUs that is a tenth filled costs most of a whole one, and smaller tiles for all of the columns
// are the slower ones.  Taken where the two estimates together are 5% less than the one launch's: at 108 sizes drawn, on four
// GPUs, 0.90 to 0.92 of one launch on average and 1.02 at most (us, one launch / two: 2048 x 8512 x 2048 94.9 / 76.3, 3001 x 7312 x 2048
// 102.9 / 91.3, 2701 x 12096 x 3520 232 / 194).  Whole rounds of 256 x 128 tiles in turns gain nothing: 0.96 to 1.03 on average at 48.
inline uint64_t dense_first_columns(uint32_t m, uint64_t columns, uint32_t k, uint32_t cus) {
  const uint64_t tiles_m = ((uint64_t)m + 255) / 256, tiles_n = (columns + 255) / 256;
  const uint64_t whole = tiles_m * tiles_n / cus * cus / tiles_m;  // tile columns of whole rounds
  if (k < staggered_from_k(DenseTile::k256x256) || whole == 0 || tiles_m * tiles_n % cus == 0 || whole * 256 >= columns) return 0;
  float one = 0.0f, rest = 0.0f;
  dense_product_tile(m, columns, k, cus, &one);
  dense_product_tile(m, columns - whole * 256, k, cus, &rest);
  return staggered_time(kStaggeredTimes[0], whole * tiles_m, columns, k, cus) + rest < 0.95f * one ? whole * 256 : 0;
}

}  // namespace llmopt
