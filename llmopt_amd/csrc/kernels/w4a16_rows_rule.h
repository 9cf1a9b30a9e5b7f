// Which W4A16 products take the small tiles of w4a16_rows.hip, and which tile: rules on sizes alone (and the number of
// compute units), without HIP, so that a host test can ask them.
#pragma once

#include <stdint.h>

namespace llmopt {

// Rows by columns of a workgroup's tile; kNone: another kernel (the matrix-core GEMV's row groups, or the 128 x 128 and
// larger tiles of w4a16_gemm.hip).
enum class RowsTile { kNone, k32x32, k32x64, k32x64Deep, k32x64Long, k64x64, k64x128, k96x128 };

// The matrix-core GEMV: rows of one group, and the longest K that one workgroup covers.
constexpr uint32_t kRowGroup = 8, kRowGroupK = 4096;
// More rows than a group, as groups of one grid: small matrices, whose weights every group decodes again.
inline bool row_groups_fit(uint32_t m, uint64_t columns, uint32_t k) {
  return m > kRowGroup && m <= 128 && k <= kRowGroupK && columns * k / 2 <= (4u << 20);
}

constexpr uint32_t kRowsLdsBytes = 160 * 1024;

// Scales of a tile in LDS: blocks of eight columns by eight groups, a dword each.
constexpr uint32_t scale_lds_bytes(uint32_t columns, uint32_t groups) { return columns / 8 * ((groups + 7) / 8) * 256; }

template <int ROWS, int CT, int P, int STAGES>
constexpr uint32_t rows_lds_bytes(uint32_t k) {
  const uint32_t ring = STAGES * (ROWS * P * 128 + CT * 32 * P * 32), sums = P * ROWS * CT * 32 * 4;
  return scale_lds_bytes(CT * 32, k / 64) + (ring > sums ? ring : sums);
}

// Rows, weights and norm weights of a whole K (w4a16_normed_rows_kernel), whose lanes hold a piece of every group.  Up to twelve groups:
// LDS has room for 24, but from thirteen on the copies that no product covers take what the norm's launch does.  us a call, norm
// apart / in the tile: QKV 90 x 576 x (576, 192) 11.4 / 9.6, 700 x 576 13.5 / 12.8, 200 x 768 x (768, 256) 11.5 / 11.1; pairs 64 x 576 x 1536
// 10.2 / 8.7, 140 x 768 x 801 11.1 / 9.5; beyond: QKV 100 x 1024 x (768, 256) 11.1 / 12.1, 128 x 1024 x (1024, 256) 11.1 / 12.2, pairs 100 x
// 1024 x 1024 10.6 / 10.9, 128 x 960 x 1024 11.0 / 10.7.
constexpr uint32_t kNormedGroups = 12;
template <int ROWS, int CT, int P>
constexpr uint32_t normed_rows_lds_bytes(uint32_t k) {
  const uint32_t groups = k / 64, sums = P * ROWS * CT * 32 * 4;
  const uint32_t whole = ROWS * groups * 128 + CT * 32 * ((groups + 1) / 2) * 64 + (groups + 7) / 8 * 1024;
  return scale_lds_bytes(CT * 32, groups) + (whole > sums ? whole : sums);
}

// The matrix-core GEMV's row groups are the better ones while they are few: up to two workgroups a CU, counted as eight
// rows by sixteen columns, of which a gated pair has both matrices in one.  The tiles' shortest launch is longer than
// theirs, more so with a long K; a third workgroup on a CU adds a whole round to them.  Each call behind the launch that
// writes its activations, us (m x K x n, GEMV / tiles):
// at 512 workgroups and below: 64 x 1024 x 1024 6.1 / 6.3, 32 x 2048 x 2048 7.2 / 8.1, 64 x 4096 x 1024 9.2 / 10.8,
// 16 x 2048 x 4096 7.1 / 8.0, 80 x 3072 x 768 8.2 / 9.4; pairs 64 x 1024 x 1024 6.7 / 7.0, 32 x 2048 x 2048 8.3 / 9.4,
// 56 x 1536 x 576 6.8 / 8.5, 64 x 4096 x 1024 11.9 / 13.4, 128 x 2048 x 512 8.8 / 9.7;
// above: 72 x 1024 x 1024 7.0 / 6.3, 33 x 2048 x 2048 8.3 / 8.0, 72 x 4096 x 1024 12.3 / 11.0, 96 x 3072 x 768 10.3 / 9.6;
// pairs 72 x 1024 x 1024 7.9 / 7.1, 40 x 2048 x 2048 10.8 / 9.5, 128 x 1536 x 576 11.2 / 8.8.
// Up to K = 512 a tile's launch is as short: there, and for the three matrices of QKV, whose groups are three launches'
// worth, the line is 48k outputs (pairs 64 x 512 x 1024 6.0 / 5.9, 33 x 512 x 2048 6.5 / 5.9).
constexpr uint64_t kRowGroupOutputs = 49152;

inline bool row_groups_few(uint32_t m, uint32_t n, uint32_t k, uint32_t cus) {
  return k > 512 && (uint64_t)((m + kRowGroup - 1) / kRowGroup) * ((n + 15) / 16) <= 2ull * cus;
}

// (The copies name a tile's bytes by 32-bit offsets from its first row.)
inline bool rows_wanted(uint32_t m, uint64_t columns, uint32_t k, bool few) {
  if (m <= kRowGroup || k > (1u << 24)) return false;
  return !(row_groups_fit(m, columns, k) && (few || m * columns <= kRowGroupOutputs));
}

// A launch takes as long as one workgroup while each CU has at most one of them, and a workgroup the longer the larger
// its tile and K are (us, K = 576 / 2048 / 4096 / 8192, one round): 32 x 32 4.1 / 6.1 / 8.8 / 13.7, 32 x 64 4.6 / 7.8 /
// 11.3 / 21, 64 x 64 5.9 / 10.3 / 16.4 / 29, 64 x 128 7.1 / 14.9 / 25.7 / 47, 96 x 128 9.5 / 18.6 / 32.4.  So: the smallest
// tile that needs one round, and the large tiles once even 96 x 128 would need a second one.  Measured against those, us (m, K,
// n):
// 24 x 4096 x 14336 13.3 / 30.8; 24 x 4096 x 4096 8.7 / 16.7; 64 x 14336 x 4096 23.5 / 38.5; 128 x 4096 x 4096 11.8 / 17.4;
// 200 x 4096 x 4096 16.9 / 21.4; 512 x 4096 x 4096 28 / 33; 1024 x 2048 x 2048 16.5 / 28.3; 700 x 576 x 576 5.3 / 9.5;
// 700 x 1536 x 576 7.0 / 13.7; 700 x 576 x 1536 7.4 / 9.5; beyond: 200 x 4096 x 14336 53.6 / 43.5, 700 x 8192 x 2048 47 / 42.
// At the line the small tiles are not the faster ones, but the more exact ones: the large tiles round q * s to half, 2.8e-4
// off float64 for 2.1e-4.  Where 64 x 128 would begin a second round and 96 x 128 is one, us 64 x 128 / 96 x 128 / large: 700 x
// 576 x 3072 11.3 / 9.5 / 10.3, 900 x 1024 x 3072 14.4 / 12.0 / 12.1, 288 x 2048 x 7680 22.2 / 19.0 / 20.0, 700 x 4096 x 3072
// 49.4 / 32.3 / 33.9, 540 x 4096 x 4096 49.1 / 32.6 / 34.0.  A long K that the large tiles split over workgroups while
// half the CUs have none of them, 300 x 3072 x 4096 22.3 / 21.4, 300 x 4096 x 4096 28.8 / 28.0, 200 x 6144 x 6144 42.1 /
// 38.7, 600 x 6144 x 2048 42.5 / 32.6.
// Beyond K = 6144 the tiles of 64 rows fit LDS up to 8192 and would win where they are one round and the large tiles pad their
// rows, not where those fill: large tiles / 64-row tiles 48 x 7168 x 14336 44.0 / 28.3, 48 x 8192 x 14336 49.4 / 32.4, 128 x
// 7168 x 8192 31.8 / 29.0, 512 x 7168 x 2048 30.4 / 28.4, 256 x 8192 x 4096 32.2 / 32.4, 200 x 7168 x 6144 43.9 / 47.9, 200 x
// 8192 x 6144 47.9 / 52.9.  They have not been taken there.
// With few steps (K < 1536) three workgroups of the shallow 32 x 64 ring share a CU: two rounds of it are still fast.
inline RowsTile rows_tile(uint32_t m, const uint32_t *n, uint32_t matrices, uint32_t k, uint32_t cus) {
  auto rounds = [&](uint32_t rows, uint32_t columns) {
    uint64_t tiles = 0;
    for (uint32_t i = 0; i < matrices; ++i) tiles += (n[i] + columns - 1) / columns;
    return (double)(tiles * ((m + rows - 1) / rows)) / cus;
  };
  if (rounds(32, 32) <= 1 && rows_lds_bytes<32, 1, 8, 3>(k) <= kRowsLdsBytes) return RowsTile::k32x32;
  if (k < 1536) {
    if (rounds(32, 64) <= 2) return RowsTile::k32x64;
  } else if (rounds(32, 64) <= 1) {
    if (rows_lds_bytes<32, 2, 8, 3>(k) <= kRowsLdsBytes) return RowsTile::k32x64Deep;
    if (rows_lds_bytes<32, 2, 4, 4>(k) <= kRowsLdsBytes) return RowsTile::k32x64Long;
  }
  if (k >= 1536 && k <= 6144 && rounds(64, 64) <= 1) return RowsTile::k64x64;
  if (k <= 6144 && rounds(64, 128) <= 1) return RowsTile::k64x128;
  if (k <= 6144 && rounds(96, 128) <= 1) return RowsTile::k96x128;
  if (k <= 6144 && rounds(64, 128) <= 1.125) return RowsTile::k64x128;  // (rows that 96 divides no better than 64)
  return RowsTile::kNone;
}

inline RowsTile linear_rows_tile(uint32_t m, uint32_t n, uint32_t k, uint32_t cus) {
  return rows_wanted(m, n, k, row_groups_few(m, n, k, cus)) ? rows_tile(m, &n, 1, k, cus) : RowsTile::kNone;
}

inline RowsTile qkv_rows_tile(uint32_t m, const uint32_t *n, uint32_t k, uint32_t cus) {
  return rows_wanted(m, (uint64_t)n[0] + n[1] + n[2], k, false) ? rows_tile(m, n, 3, k, cus) : RowsTile::kNone;
}

// QKV with the rotation and the Q8 pack: a tile of whole heads.  Where the rule takes half a head's columns, the 64-column
// one, whose few microseconds more are less than another launch.
inline RowsTile pack_rows_tile(uint32_t m, const uint32_t *n, uint32_t k, uint32_t cus) {
  const RowsTile tile = qkv_rows_tile(m, n, k, cus);
  if (tile != RowsTile::k32x32) return tile;
  if (k < 1536) return RowsTile::k32x64;
  if (rows_lds_bytes<32, 2, 8, 3>(k) <= kRowsLdsBytes) return RowsTile::k32x64Deep;
  return rows_lds_bytes<32, 2, 4, 4>(k) <= kRowsLdsBytes ? RowsTile::k32x64Long : RowsTile::kNone;
}

// A gated pair, by output columns (half of a tile's).  The large tiles take two accumulator sets, so the
// small ones win for longer: us (m, K, n) 24 x 4096 x 14336 20.4 / 61.7, 64 x 4096 x 4096 12.6 / 58, 64 x 8192 x 2048
// 26 / 108, 128 x 4096 x 14336 55 / 64 (two rounds), 512 x 2048 x 2048 15.9 / 31.8, 1024 x 2048 x 2048 26.3 / 34.4,
// 700 x 576 x 1536 10.9 / 16.0; beyond: 200 x 4096 x 14336 105 / 78, 2048 x 2048 x 2048 49 / 46.  Where 96 x 128 is one round and
// 64 x 128 is not, us 64 x 128 / 96 x 128: 700 x 576 x 1536 10.6 / 9.0, 900 x 1024 x 1536 13.6 / 11.4, 540 x 2048 x 2048 21.7 /
// 18.0, 700 x 4096 x 1536 50.6 / 31.4.
inline RowsTile gated_rows_tile(uint32_t m, uint32_t n, uint32_t k, uint32_t cus) {
  if (!rows_wanted(m, 2ull * n, k, row_groups_few(m, n, k, cus))) return RowsTile::kNone;
  auto rounds = [&](uint32_t rows, uint32_t columns) {
    return (double)((uint64_t)((n + columns - 1) / columns) * ((m + rows - 1) / rows)) / cus;
  };
  if (rounds(32, 32) <= 1) {
    if (k < 1536) return RowsTile::k32x64;
    if (rows_lds_bytes<32, 2, 8, 3>(k) <= kRowsLdsBytes) return RowsTile::k32x64Deep;
    if (rows_lds_bytes<32, 2, 4, 4>(k) <= kRowsLdsBytes) return RowsTile::k32x64Long;
  }
  if (rounds(64, 32) <= 1 && rows_lds_bytes<64, 2, 4, 3>(k) <= kRowsLdsBytes) return RowsTile::k64x64;
  if (rounds(32, 32) <= 2 && k <= 8192) return RowsTile::k32x64;
  if (rounds(64, 64) > 1 && rounds(96, 64) <= 1 && rows_lds_bytes<96, 4, 2, 2>(k) <= kRowsLdsBytes) return RowsTile::k96x128;
  if (rounds(64, 64) <= 2 && rows_lds_bytes<64, 4, 2, 2>(k) <= kRowsLdsBytes) return RowsTile::k64x128;
  return RowsTile::kNone;
}

// Logits of rows / 2 tokens (a hi and a lo row each).  The tile is the one above while the launch is about one round, and
// beyond, where the 128 x 128 tiles have no float32 results, the one that decodes the weights least often of those whose
// scales fit LDS beside the ring.  With a long K a few rows stay with the matrix-core GEMV, which streams the weights better
// than a tile that is mostly padding.  Head with its argmax behind the launch that writes its rows, us, GEMV / tiles (tokens,
// K, n): to the GEMV 8 x 2048 x 32000 44.1 / 48.7, 12 x 2048 x 32000 47.1 / 48.9 (64 x 128 tiles), 8 x 3072 x 32000 56 / 62,
// 8 x 4096 x 16384 52.6 / 62.6, 12 x 4096 x 32000 77 / 82, 8 x 8192 x 8192 82 / 90, 16 x 2048 x 2048 27.1 / 28.1 (two GEMV
// workgroups a CU); to the tiles 5 x 576 x 49152 32.9 / 24.6, 32 x 576 x 49152 61 / 31, 12 x 1536 x 32000 42.1 / 38.0,
// 12 x 2048 x 16384 39.6 / 37.0, 16 x 2048 x 32000 56.7 / 49.0, 12 x 4096 x 16384 64.8 / 62.4, 20 x 4096 x 32000 110 / 83,
// 64 x 4096 x 32000 197 / 107, 16 x 8192 x 8192 107 / 90.  A tile's rows are a row of the grid, which has at most 65536.
inline RowsTile logits_rows_tile(uint32_t rows, uint32_t n, uint32_t k, uint32_t cus) {
  if (!rows_wanted(rows, n, k, k >= 1280 && rows <= 32 && row_groups_few(rows, n, k, cus))) return RowsTile::kNone;
  const RowsTile small = rows_tile(rows, &n, 1, k, cus);
  if (k >= 2048 && (rows <= 16 || (rows <= 24 && small == RowsTile::k64x128))) return RowsTile::kNone;
  if (small != RowsTile::kNone) return small;
  if (k >= 1536 && rows <= 24) return RowsTile::kNone;
  if (rows > 32 && rows <= 65536 * 64 && rows_lds_bytes<64, 4, 2, 2>(k) <= kRowsLdsBytes) return RowsTile::k64x128;
  if (rows <= 65536 * 32 && rows_lds_bytes<32, 2, 4, 2>(k) <= kRowsLdsBytes) return RowsTile::k32x64;
  return RowsTile::kNone;
}

// Whether a tile normalises its rows itself: tiles of 32 rows and at most kNormedGroups groups of K, in one round of workgroups.
inline bool normed_rows(RowsTile tile, uint32_t m, const uint32_t *n, uint32_t matrices, uint32_t k, uint32_t cus) {
  if (tile != RowsTile::k32x64 || k > kNormedGroups * 64) return false;
  uint64_t tiles = 0;
  for (uint32_t i = 0; i < matrices; ++i) tiles += ((uint64_t)n[i] + 63) / 64;
  return tiles * ((m + 31) / 32) <= (uint64_t)cus * (kRowsLdsBytes / normed_rows_lds_bytes<32, 2, 4>(k));
}

}  // namespace llmopt
