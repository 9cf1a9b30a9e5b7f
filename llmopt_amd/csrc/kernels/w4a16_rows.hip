// W4A16 products of a batch's rows (more than the streaming GEMVs take, fewer than a prompt's) and of prompts over small
// matrices: tiles of 32 to 96 activation rows by 32, 64 or 128 weight columns (w4a16_rows_rule.h), so that the launch has
// about a workgroup per CU where 128 x 128 tiles leave most of them empty or pad most of their rows.
//
// What bounds it at many rows of K: the weights from HBM (31 MB at 4096 x 14336: 6.5 us at a copy's rate) and the
// activation rows, which every workgroup reads again, from L2; at a CU's rate of filling LDS (about 80 bytes a
// nanosecond) 32 rows take 3 us and 64 rows 6 us of their own.  With a short K, the start of a launch and two or three
// trips to memory.
//
//  * A workgroup is CT x P waves.  A step covers P scale groups (64 K values each) of the tile's rows and columns; wave
//    (ct, p) multiplies group p of the step into the 32 columns ct.  The waves that share columns split K this way at the
//    finest grain, so a step's requests are whole lines of every row, and their sums meet once, at the end, in LDS.
//  * Both operands go global -> LDS as direct copies, a ring of STAGES steps, waited for by count, one barrier a step.
//    16-byte pieces are XOR-ed by the row, so that the rows an operand read touches lie in different banks.
//  * A lane of the 32 x 32 x 16 product holds 32 K values (16 bytes) of one weight row and its partner lane the other
//    half of the same scale group: four products a group, on exact integers, and the group's fp16 scale is one float32
//    multiply-add per sum, as in the GEMVs (the 128 x 128 tiles round q * s to half).
//  * The scales of the tile are copied to LDS ahead of everything else (a dword each).
//
// Measured at 24 x 4096 x 14336 (us): 13.3 (128 x 128 tiles 27 to 31), of which 4.9 the launch's start, first trip to memory and
// epilogue; the copies alone take 9.3 and the products alone 10.6 of the same launch: 85 vector instructions a wave and
// step (52 of them the decode) beside 24 KB of copies.  Tried without gain: operands read a step ahead of their use,
// two column blocks a wave, a start of the walk over K that differs by workgroup, deeper rings.
#include <algorithm>
#include <type_traits>

#include "kernels.h"
#include "kernels_internal.h"
#include "w4_common.h"
#include "w4a16_rows_rule.h"

namespace llmopt {
namespace {

struct RowsParams {
  const uint16_t *x;
  uint32_t m, k;
  // One matrix, the two of a gated pair (tile columns alternate), or several that multiply the same rows: their column
  // tiles follow each other.
  const uint8_t *w[3];
  const uint16_t *s[3];
  uint16_t *y[3];
  uint32_t n[3];
  uint32_t tiles[3];
  uint32_t segments;
  const uint16_t *addend;
  uint32_t addend_stride;
  float *pairs;  // [m / 2, n]: in place of y, the float32 sums of rows 2r and 2r + 1
};

// A QKV launch whose queries and keys are rotated and whose keys and values also go to their tokens' Q8 pool slots, in
// the arithmetic of launch_rotary_qk_pack: heads of 64 columns, one sequence.  y[0] and y[1] are then the rotated
// outputs [head, token, 64].  One layer's launch at 700 x 576 x (576, 192, 192): 8.2 us where the projection and the
// rotation with the pack take 7.0 + 5.5, most of either the start of a launch.
struct PackParams : RowsParams {
  const uint16_t *cosine, *sine;  // [token, 64]
  const uint32_t *slots;
  uint8_t *pool;
  uint32_t token_stride, token_elements, segment_offset[2];
};

// base + offset (bytes, per lane) to consecutive LDS places: sixteen bytes a lane ...
__device__ __forceinline__ void copy16_to_lds(const void *base, uint32_t offset, uint32_t lds_address) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(offset), "s"(base), "s"(lds_address) : "memory");
}
// ... or two, stored as a dword.
__device__ __forceinline__ void copy2_to_lds(const void *base, uint32_t offset, uint32_t lds_address) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_ushort %0, %1" : : "v"(offset), "s"(base), "s"(lds_address) : "memory");
}

// Eight weights of a dword as exact halves in K order.
__device__ __forceinline__ h8_t w4_exact_natural(uint32_t word) {
  const W4Pairs q = w4_decode_pairs(word);
  const uint32_t p04 = as_u32(q.p04), p15 = as_u32(q.p15), p26 = as_u32(q.p26), p37 = as_u32(q.p37);
  uint4 packed;
  packed.x = __builtin_amdgcn_perm(p15, p04, 0x05040100u);
  packed.y = __builtin_amdgcn_perm(p37, p26, 0x05040100u);
  packed.z = __builtin_amdgcn_perm(p15, p04, 0x07060302u);
  packed.w = __builtin_amdgcn_perm(p37, p26, 0x07060302u);
  return __builtin_bit_cast(h8_t, packed);
}

// What a workgroup's lanes need of their place in the launch.
struct TileLane {
  uint32_t segment, n, m0, n0;  // the matrix, its columns, the tile's first row and column
  int part, column, half;       // of the wave's K groups; of the tile; which half of a block's rows
};

// The end of a tile: the waves' sums meet in LDS, [part][row][column], added in the order of the parts, and go out.
template <int ROWS, int CT, int P, bool DUAL, class Params>
__device__ __forceinline__ void finish_rows(const Params &p, const f16x_t (&acc)[ROWS / 32], const TileLane &at_tile, float *sums) {
  constexpr bool PACK = std::is_same_v<Params, PackParams>;
  constexpr int WAVES = CT * P, COLUMNS = CT * 32, RT = ROWS / 32;
  const int tid = threadIdx.x, part = at_tile.part, column = at_tile.column, half = at_tile.half;
  const uint32_t segment = at_tile.segment, n = at_tile.n, m0 = at_tile.m0, n0 = at_tile.n0;
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __syncthreads();
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int row = r * 32 + (i >> 2) * 8 + half * 4 + (i & 3);
      sums[(part * ROWS + row) * COLUMNS + column] = acc[r][i];
    }
  __syncthreads();
  constexpr int OUT = DUAL ? COLUMNS / 2 : COLUMNS, QUADS = ROWS * OUT / 4;
  if constexpr (PACK) {
    typedef uint16_t u16x4_t __attribute__((ext_vector_type(4), aligned(2)));
    typedef uint32_t any_u32_t __attribute__((aligned(1)));
    // a head of a row is sixteen neighbouring lanes
    for (int q = tid; q < QUADS; q += WAVES * 64) {
      const uint32_t row = q / (OUT / 4), c = q % (OUT / 4) * 4, at = m0 + row;
      if (at >= p.m || n0 + c >= n) continue;
      const uint32_t head = (n0 + c) / 64, d = c % 64;
      f4_t value = {0.f, 0.f, 0.f, 0.f}, other = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < P; ++k) {
        value += *reinterpret_cast<const f4_t *>(sums + (k * ROWS + row) * COLUMNS + c);
        other += *reinterpret_cast<const f4_t *>(sums + (k * ROWS + row) * COLUMNS + (c ^ 32));
      }
      u16x4_t out;
      float wide[4];
      if (segment < 2) {
        const u16x4_t cosine = *reinterpret_cast<const u16x4_t *>(p.cosine + (size_t)at * 64 + d);
        const u16x4_t sine = *reinterpret_cast<const u16x4_t *>(p.sine + (size_t)at * 64 + d);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const _Float16 turned = rotate_half_value((_Float16)value[e], (_Float16)other[e], __builtin_bit_cast(_Float16, (uint16_t)cosine[e]),
                                                    __builtin_bit_cast(_Float16, (uint16_t)sine[e]), d < 32);
          out[e] = __builtin_bit_cast(uint16_t, turned);
          wide[e] = (float)turned;
        }
        *reinterpret_cast<u16x4_t *>(p.y[segment] + ((size_t)head * p.m + at) * 64 + d) = out;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          out[e] = float_to_half_bits(value[e]);
          wide[e] = half_bits_to_float(out[e]);
        }
        *reinterpret_cast<u16x4_t *>(p.y[2] + (size_t)at * n + n0 + c) = out;
      }
      if (segment == 0) continue;
      float maximum = fmaxf(fmaxf(fabsf(wide[0]), fabsf(wide[1])), fmaxf(fabsf(wide[2]), fabsf(wide[3])));
#pragma unroll
      for (int lanes = 1; lanes < 16; lanes *= 2) maximum = fmaxf(maximum, __shfl_xor(maximum, lanes, 64));
      uint16_t stored;
      uint32_t packed = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) packed |= (uint32_t)(uint8_t)q8_quantize_by(wide[e], maximum, &stored) << (8 * e);
      uint8_t *slot = p.pool + (size_t)p.slots[at] * p.token_stride;
      const uint32_t offset = p.segment_offset[segment - 1] + head * 64;
      *reinterpret_cast<any_u32_t *>(slot + offset + d) = packed;
      if (d == 0) reinterpret_cast<uint16_t *>(slot + p.token_elements)[offset / 64] = stored;
    }
    return;
  }
  if (!DUAL && p.pairs != nullptr) {
    const bool whole = (n & 3) == 0 && (reinterpret_cast<uintptr_t>(p.pairs) & 15) == 0;
    for (int q = tid; q < QUADS / 2; q += WAVES * 64) {
      const uint32_t row = q / (OUT / 4) * 2, c = q % (OUT / 4) * 4, at = m0 + row;
      if (at >= p.m || n0 + c >= n) continue;
      f4_t value[2];
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        value[r] = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < P; ++k) value[r] += *reinterpret_cast<const f4_t *>(sums + (k * ROWS + row + r) * COLUMNS + c);
      }
      const f4_t sum = value[0] + value[1];
      float *to = p.pairs + (size_t)(at / 2) * n + n0 + c;
      if (whole) {
        *reinterpret_cast<f4_t *>(to) = sum;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n0 + c + e < n) to[e] = sum[e];
      }
    }
    return;
  }
  uint16_t *y = p.y[segment];
  const bool whole = (n & 3) == 0 && (reinterpret_cast<uintptr_t>(y) & 7) == 0;
  for (int q = tid; q < QUADS; q += WAVES * 64) {
    const uint32_t row = q / (OUT / 4), c = q % (OUT / 4) * 4, at = m0 + row;
    if (at >= p.m || n0 + c >= n) continue;
    // of a pair: 32 gate columns, then the 32 up columns of the same outputs
    const uint32_t from = DUAL ? (c >> 5) * 64 + (c & 31) : c;
    f4_t value = {0.f, 0.f, 0.f, 0.f}, up = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < P; ++k) {
      value += *reinterpret_cast<const f4_t *>(sums + (k * ROWS + row) * COLUMNS + from);
      if (DUAL) up += *reinterpret_cast<const f4_t *>(sums + (k * ROWS + row) * COLUMNS + from + 32);
    }
    uint16_t out[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float v = value[e];
      if (DUAL) v = v / (1.0f + __expf(-v)) * up[e];
      if (!DUAL && p.addend != nullptr && n0 + c + e < n)
        v += half_bits_to_float(p.addend[(size_t)at * p.addend_stride + n0 + c + e]);
      out[e] = float_to_half_bits(v);
    }
    uint16_t *to = y + (size_t)at * n + n0 + c;
    if (whole) {
      *reinterpret_cast<ushort4 *>(to) = ushort4{out[0], out[1], out[2], out[3]};
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n0 + c + e < n) to[e] = out[e];
    }
  }
}


template <int ROWS, int CT, int P, int STAGES, bool DUAL, class Params>
__global__ __launch_bounds__(CT *P * 64) void w4a16_rows_kernel(Params p) {
  constexpr bool PACK = std::is_same_v<Params, PackParams>;
  static_assert(!PACK || (!DUAL && CT % 2 == 0), "whole heads in a tile");
  constexpr int WAVES = CT * P, COLUMNS = CT * 32, STEP = P * 64;
  static_assert(ROWS % 32 == 0, "whole blocks of rows");
  constexpr int RT = ROWS / 32;                             // 32-row blocks of a wave
  constexpr int X_PIECES = STEP / 8, W_PIECES = STEP / 32;  // 16-byte pieces of a row and step
  constexpr int X_BYTES = ROWS * X_PIECES * 16, W_BYTES = COLUMNS * W_PIECES * 16, STAGE_BYTES = X_BYTES + W_BYTES;
  constexpr int X_COPIES = X_BYTES / 1024 / WAVES, COPIES = X_COPIES + 1;  // of a wave and step
  static_assert(X_BYTES == X_COPIES * WAVES * 1024 && W_BYTES == WAVES * 1024, "a step divides over the waves");
  static_assert(!DUAL || CT % 2 == 0, "gate and up columns of an output lie in one tile");
  extern __shared__ __attribute__((aligned(16))) unsigned char rows_lds[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ct = wave / P, part = wave % P;
  const uint32_t groups = p.k / 64, steps = (groups + P - 1) / P;

  uint32_t segment = 0, tile = blockIdx.x;
  if (!DUAL)
    while (segment + 1 < p.segments && tile >= p.tiles[segment]) tile -= p.tiles[segment++];
  const uint32_t n = p.n[segment], m0 = blockIdx.y * ROWS;
  const uint32_t n0 = tile * (DUAL ? COLUMNS / 2 : COLUMNS);
  // Of a tile column: its row in the matrix, from the tile's first one (columns past n are never stored).  The 32-column
  // blocks of a pair's tile alternate between gate and up.
  auto weight_row = [&](uint32_t column) __attribute__((always_inline)) {
    return min(DUAL ? (column >> 6) * 32 + (column & 31) : column, n - 1 - n0);
  };
  auto matrix_of = [&](uint32_t column) __attribute__((always_inline)) { return DUAL ? (column >> 5) & 1 : segment; };

  const uint32_t scale_bytes = scale_lds_bytes(COLUMNS, groups);
  const uint32_t lds_base = (uint32_t)(size_t)(__attribute__((address_space(3))) unsigned char *)rows_lds;
  const uint32_t ring = lds_base + scale_bytes;
  const uint32_t group_blocks = (groups + 7) / 8;
  for (uint32_t block = wave; block < COLUMNS / 8 * group_blocks; block += WAVES) {
    const uint32_t column = block / group_blocks * 8;
    const uint16_t *scales = p.s[matrix_of(column)] + (size_t)n0 * groups;
    const uint32_t row = weight_row(column + (lane & 7)), group = min(block % group_blocks * 8 + (lane >> 3), groups - 1);
    copy2_to_lds(scales, (row * groups + group) * 2, lds_base + block * 256);
  }

  // Copies of a step: lane l fills consecutive 16-byte places; the piece it fetches is the one that the swizzle puts there.
  const uint8_t *x_base = reinterpret_cast<const uint8_t *>(p.x + (size_t)m0 * p.k);
  uint32_t x_row[X_COPIES], x_at[X_COPIES];  // bytes
#pragma unroll
  for (int c = 0; c < X_COPIES; ++c) {
    const uint32_t place = (wave * X_COPIES + c) * 64 + lane, row = place / X_PIECES;
    x_row[c] = min(row, p.m - 1 - m0) * p.k * 2;
    x_at[c] = (place % X_PIECES ^ (row & 15)) * 16;
  }
  auto w_twist = [](uint32_t row) __attribute__((always_inline)) {
    return W_PIECES >= 16 ? row & 15 : W_PIECES == 8 ? (row >> 1) & 7 : (row >> 2) & 3;
  };
  const uint32_t w_place = wave * 64 + lane, w_column = w_place / W_PIECES;
  const uint8_t *w_base = p.w[matrix_of(wave * 64 / W_PIECES)] + (size_t)n0 * (p.k / 2);
  const uint32_t w_row = weight_row(w_column) * (p.k / 2), w_at = (w_place % W_PIECES ^ w_twist(w_column)) * 16;
  auto request = [&](uint32_t step) __attribute__((always_inline)) {
    const uint32_t stage = ring + step % STAGES * STAGE_BYTES, k0 = step * STEP;
    const uint8_t *x = x_base + (size_t)k0 * 2, *w = w_base + k0 / 2;
    if (k0 + STEP <= p.k) {
      copy16_to_lds(w, w_row + w_at, stage + X_BYTES + wave * 1024);
#pragma unroll
      for (int c = 0; c < X_COPIES; ++c) copy16_to_lds(x, x_row[c] + x_at[c], stage + (wave * X_COPIES + c) * 1024);
    } else {  // the end of the rows: their last pieces again, which nothing multiplies
      copy16_to_lds(w, w_row + min(w_at, (p.k - k0) / 2 - 16), stage + X_BYTES + wave * 1024);
#pragma unroll
      for (int c = 0; c < X_COPIES; ++c)
        copy16_to_lds(x, x_row[c] + min(x_at[c], (p.k - k0) * 2 - 16), stage + (wave * X_COPIES + c) * 1024);
    }
  };

  f16x_t acc[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[r][i] = 0.0f;

  const int column = ct * 32 + (lane & 31), half = lane >> 5;
  const uint32_t x_read_row = lane & 31;
  const uint32_t w_read = X_BYTES + (column * W_PIECES + ((part * 2 + half) ^ w_twist(column))) * 16;
  uint32_t x_read[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) x_read[j] = (x_read_row * X_PIECES + ((part * 8 + half * 4 + j) ^ (x_read_row & 15))) * 16;
  const uint32_t *scale_read = reinterpret_cast<const uint32_t *>(rows_lds) + (column >> 3) * group_blocks * 64 + (column & 7);
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < (int)steps) request(s);
  for (uint32_t s = 0; s < steps; ++s) {
    // this step has landed once only the copies of the STAGES - 2 steps behind it are under way
    if (s + STAGES - 2 < steps) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"((STAGES - 2) * COPIES) : "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (s + STAGES - 1 < steps) request(s + STAGES - 1);  // into the place of the step before, which every wave has read
    const uint32_t group = s * P + part;
    if (group >= groups) continue;  // (the same for the whole wave, and its last step)
    const unsigned char *stage = rows_lds + scale_bytes + s % STAGES * STAGE_BYTES;
    const u32x4_t packed = *reinterpret_cast<const u32x4_t *>(stage + w_read);
    h8_t x[RT][4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < RT; ++r)
        x[r][j] = *reinterpret_cast<const h8_t *>(stage + x_read[j] + r * 32 * X_PIECES * 16);
    const float scale = half_bits_to_float((uint16_t)scale_read[(group >> 3) * 64 + (group & 7) * 8]);
    f16x_t sum[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int i = 0; i < 16; ++i) sum[r][i] = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const h8_t w = w4_exact_natural(packed[j]);
#pragma unroll
      for (int r = 0; r < RT; ++r) sum[r] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[r][j], w, sum[r], 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[r][i] = fmaf(scale, sum[r][i], acc[r][i]);
  }

  finish_rows<ROWS, CT, P, DUAL>(p, acc, {segment, n, m0, n0, part, column, half}, reinterpret_cast<float *>(rows_lds + scale_bytes));
}

// The value of another lane of the same sixteen.
template <int CONTROL>
__device__ __forceinline__ float lane_of(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CONTROL, 0xf, 0xf, true));
}

// half(x * gain * inverse) (FIRST) or half(x * inverse * gain) of two values, every product rounded to float32 and the last one
// then to half.  Halves are read where they lie: without their conversions it is 3.5 instructions a value for 5.5.  (A zero may
// lose its sign, which no sum shows.)
template <bool FIRST>
__device__ __forceinline__ uint32_t normed_pair(uint32_t x, uint32_t gain, float inverse) {
  float low, high;
  if (FIRST) {
    asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel_hi:[1,1,0]" : "=v"(low) : "v"(x), "v"(gain));
    asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[1,1,0] op_sel_hi:[1,1,0]" : "=v"(high) : "v"(x), "v"(gain));
    asm("v_mul_f32 %0, %1, %2" : "=v"(low) : "v"(low), "v"(inverse));  // (a product that the compiler sees it rounds to half at once)
    asm("v_mul_f32 %0, %1, %2" : "=v"(high) : "v"(high), "v"(inverse));
  } else {
    float turned[2];
    asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel_hi:[1,0,0]" : "=v"(turned[0]) : "v"(x), "v"(inverse));
    asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(turned[1]) : "v"(x), "v"(inverse));
    asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel_hi:[0,1,0]" : "=v"(low) : "v"(turned[0]), "v"(gain));
    asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[0,1,0] op_sel_hi:[0,1,0]" : "=v"(high) : "v"(turned[1]), "v"(gain));
  }
  return (uint32_t)float_to_half_bits(low) | (uint32_t)float_to_half_bits(high) << 16;
}

// The same tiles over rows that the kernel normalises itself, for a short K (kNormedGroups) all of whose rows and weights lie in
// LDS: everything is requested at once, waves normalise the rows where they lie, eight lanes a row, and the products follow without
// a barrier between them.  The launch of the norm ahead, 3.4 us of starting and a trip to memory and back, and its boundary go.
// With 32 rows of 576 values that is the better one (QKV with rotation and pack, 700 rows: 8.0 + 3.4 us and the boundary / 11.2; a
// pair of 64 x 576 x 1536 10.2 / 8.7 a call; prompts of 64 to 900 tokens of a 30-layer transformer 1.5 to 3.5% less), with 96 rows the
// copies that no product covers cost as much (a pair of 700 x 576 x 1536: 10.8 + 3.4 / 15.6).
//
//  * Rows lie as blocks of eight rows by one scale group, 1 KB that a copy fills from whole lines, pieces XOR-ed by half the row;
//    weights as blocks of sixteen columns by two groups, pieces XOR-ed by a quarter of the column.  Operand reads of sixteen
//    lanes touch every bank once.
//  * The arithmetic is that of rms_norm_f16_rows_kernel and w4a16_rows_kernel in their order: the same values.
template <int ROWS, int CT, int P, bool DUAL, class Params>
__global__ __launch_bounds__(CT *P * 64) void w4a16_normed_rows_kernel(Params p, W4Norm norm) {
  static_assert(!std::is_same_v<Params, PackParams> || (!DUAL && CT % 2 == 0), "whole heads in a tile");
  static_assert(ROWS % 32 == 0 && (!DUAL || CT % 2 == 0), "whole blocks; gate and up columns of an output in one tile");
  constexpr int WAVES = CT * P, COLUMNS = CT * 32, RT = ROWS / 32;
  extern __shared__ __attribute__((aligned(16))) unsigned char rows_lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ct = wave / P, part = wave % P;
  const uint32_t groups = p.k / 64, pairs = (groups + 1) / 2;

  uint32_t segment = 0, tile = blockIdx.x;
  if (!DUAL)
    while (segment + 1 < p.segments && tile >= p.tiles[segment]) tile -= p.tiles[segment++];
  const uint32_t n = p.n[segment], m0 = blockIdx.y * ROWS, n0 = tile * (DUAL ? COLUMNS / 2 : COLUMNS);
  auto weight_row = [&](uint32_t column) __attribute__((always_inline)) {
    return min(DUAL ? (column >> 6) * 32 + (column & 31) : column, n - 1 - n0);
  };
  auto matrix_of = [&](uint32_t column) __attribute__((always_inline)) { return DUAL ? (column >> 5) & 1 : segment; };

  const uint32_t scale_bytes = scale_lds_bytes(COLUMNS, groups), x_bytes = ROWS * groups * 128;
  const uint32_t lds_base = (uint32_t)(size_t)(__attribute__((address_space(3))) unsigned char *)rows_lds;
  // rows: lane l fetches the piece that the swizzle puts at place l % 8 of row l / 8
  for (uint32_t copy = wave; copy < ROWS / 8 * groups; copy += WAVES) {
    const uint32_t block = copy % (ROWS / 8), group = copy / (ROWS / 8), row = block * 8 + (lane >> 3);
    const uint16_t *x = p.x + (size_t)m0 * p.k + group * 64;
    copy16_to_lds(x, min(row, p.m - 1 - m0) * p.k * 2 + (((lane & 7) ^ ((row >> 1) & 7)) * 16),
                  lds_base + scale_bytes + (block * groups + group) * 1024);
  }
  // weights: a block's columns lie in one matrix; the second half of the last pair of an odd K is the first one again
  for (uint32_t copy = wave; copy < COLUMNS / 16 * pairs; copy += WAVES) {
    const uint32_t block = copy % (COLUMNS / 16), pair = copy / (COLUMNS / 16), first = block * 16, column = first + (lane >> 2);
    const uint8_t *w = p.w[matrix_of(first)] + (size_t)n0 * (p.k / 2);
    const uint32_t piece = (lane & 3) ^ ((column >> 2) & 3), group = min(pair * 2 + piece / 2, groups - 1);
    copy16_to_lds(w, weight_row(column) * (p.k / 2) + group * 32 + piece % 2 * 16, lds_base + scale_bytes + x_bytes + (block * pairs + pair) * 1024);
  }
  const uint32_t group_blocks = (groups + 7) / 8;
  for (uint32_t copy = wave; copy < COLUMNS / 8 * group_blocks; copy += WAVES) {
    const uint32_t block = copy % (COLUMNS / 8), eight = copy / (COLUMNS / 8), column = block * 8;
    const uint16_t *scales = p.s[matrix_of(column)] + (size_t)n0 * groups;
    const uint32_t row = weight_row(column + (lane & 7)), group = min(eight * 8 + (lane >> 3), groups - 1);
    copy2_to_lds(scales, (row * groups + group) * 2, lds_base + (block * group_blocks + eight) * 256);
  }
  const uint32_t gain_offset = x_bytes + COLUMNS / 16 * pairs * 1024;
  for (uint32_t block = wave; block * 8 < groups; block += WAVES)
    copy16_to_lds(norm.weight, min(block * 64 + lane, groups * 8 - 1) * 16, lds_base + scale_bytes + gain_offset + block * 1024);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  unsigned char *rows = rows_lds + scale_bytes;
  for (uint32_t block = wave; block < ROWS / 8; block += WAVES) {
    const uint32_t row = block * 8 + (lane >> 3), piece = (lane & 7) ^ ((row >> 1) & 7);
    unsigned char *place = rows + block * groups * 1024 + lane * 16;
    const unsigned char *gains = rows + gain_offset + piece * 16;
    u32x4_t x[kNormedGroups];
#pragma unroll
    for (uint32_t group = 0; group < kNormedGroups; ++group)
      x[group] = group < groups ? *reinterpret_cast<const u32x4_t *>(place + group * 1024) : u32x4_t{0, 0, 0, 0};
    // in the order of rms_norm_f16_rows_kernel, whose lane l has pieces l, l + 64, ..: here the lane's pieces of groups b, b + 8
    float eight[8];
#pragma unroll
    for (uint32_t b = 0; b < 8; ++b) {
      float sum = 0.0f;
#pragma unroll
      for (uint32_t group = b; group < kNormedGroups; group += 8)
        if (group < groups) {
          const h8_t v = __builtin_bit_cast(h8_t, x[group]);
#pragma unroll
          for (int e = 0; e < 8; ++e) sum += (float)v[e] * (float)v[e];
        }
      sum += lane_of<0xb1>(sum);   // neighbours
      sum += lane_of<0x4e>(sum);   // pairs
      sum += lane_of<0x141>(sum);  // halves of eight lanes
      eight[b] = sum;
    }
    const float square_sum = ((eight[0] + eight[1]) + (eight[2] + eight[3])) + ((eight[4] + eight[5]) + (eight[6] + eight[7]));
    const float inverse = rsqrtf(square_sum / (float)p.k + norm.epsilon);
#pragma unroll
    for (uint32_t group = 0; group < kNormedGroups; ++group)
      if (group < groups) {
        const u32x4_t g = *reinterpret_cast<const u32x4_t *>(gains + group * 128);
        u32x4_t y;
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = normed_pair<DUAL>(x[group][e], g[e], inverse);
        *reinterpret_cast<u32x4_t *>(place + group * 1024) = y;
      }
  }
  __syncthreads();

  f16x_t acc[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[r][i] = 0.0f;
  const int column = ct * 32 + (lane & 31), half = lane >> 5;
  const uint32_t row = lane & 31, row_twist = (row >> 1) & 7, column_twist = (column >> 2) & 3;
  const unsigned char *x_own = rows + (row >> 3) * groups * 1024 + (row & 7) * 128;
  const unsigned char *w_own = rows + x_bytes + (column >> 4) * pairs * 1024 + (column & 15) * 64;
  const uint32_t *scale_own = reinterpret_cast<const uint32_t *>(rows_lds) + (column >> 3) * group_blocks * 64 + (column & 7);
  for (uint32_t group = part; group < groups; group += P) {
    const u32x4_t packed = *reinterpret_cast<const u32x4_t *>(w_own + (group >> 1) * 1024 + (((group & 1) * 2 + half) ^ column_twist) * 16);
    h8_t x[RT][4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < RT; ++r)
        x[r][j] = *reinterpret_cast<const h8_t *>(x_own + (r * 4 * groups + group) * 1024 + ((half * 4 + j) ^ row_twist) * 16);
    const float scale = half_bits_to_float((uint16_t)scale_own[(group >> 3) * 64 + (group & 7) * 8]);
    f16x_t sum[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int i = 0; i < 16; ++i) sum[r][i] = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const h8_t w = w4_exact_natural(packed[j]);
#pragma unroll
      for (int r = 0; r < RT; ++r) sum[r] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[r][j], w, sum[r], 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[r][i] = fmaf(scale, sum[r][i], acc[r][i]);
  }
  finish_rows<ROWS, CT, P, DUAL>(p, acc, {segment, n, m0, n0, part, column, half}, reinterpret_cast<float *>(rows));
}

template <int ROWS, int CT, int P, int STAGES, bool DUAL, class Params>
hipError_t run_rows(Params &p, hipStream_t stream) {
  const auto kernel = w4a16_rows_kernel<ROWS, CT, P, STAGES, DUAL, Params>;
  const uint32_t bytes = rows_lds_bytes<ROWS, CT, P, STAGES>(p.k);
  if (bytes > kRowsLdsBytes) return hipErrorInvalidValue;
  static bool allowed[kMaxDevices] = {};
  if (hipError_t status = allow_dynamic_lds(reinterpret_cast<const void *>(kernel), kRowsLdsBytes, allowed)) return status;
  constexpr uint32_t columns = DUAL ? CT * 16 : CT * 32;
  uint32_t tiles = 0;
  for (uint32_t i = 0; i < p.segments; ++i) tiles += p.tiles[i] = (p.n[i] + columns - 1) / columns;
  kernel<<<dim3(tiles, (p.m + ROWS - 1) / ROWS), CT * P * 64, bytes, stream>>>(p);
  return hipGetLastError();
}

template <bool DUAL, class Params>
hipError_t launch_tile(RowsTile tile, Params &p, hipStream_t stream) {
  switch (tile) {
    case RowsTile::k32x32:
      if constexpr (!DUAL && std::is_same_v<Params, RowsParams>) return run_rows<32, 1, 8, 3, false>(p, stream);
      return hipErrorInvalidValue;
    case RowsTile::k32x64: return run_rows<32, 2, 4, 2, DUAL>(p, stream);
    case RowsTile::k32x64Deep: return run_rows<32, 2, 8, 3, DUAL>(p, stream);
    case RowsTile::k32x64Long: return run_rows<32, 2, 4, 4, DUAL>(p, stream);
    case RowsTile::k64x64: return run_rows<64, 2, 4, 3, DUAL>(p, stream);
    case RowsTile::k64x128: return run_rows<64, 4, 2, 2, DUAL>(p, stream);
    case RowsTile::k96x128: return run_rows<96, 4, 2, 2, DUAL>(p, stream);
    case RowsTile::kNone: break;
  }
  return hipErrorInvalidValue;
}

template <int ROWS, int CT, int P, bool DUAL, class Params>
hipError_t run_normed_rows(Params &p, const W4Norm &norm, hipStream_t stream) {
  const auto kernel = w4a16_normed_rows_kernel<ROWS, CT, P, DUAL, Params>;
  const uint32_t bytes = normed_rows_lds_bytes<ROWS, CT, P>(p.k);
  if (bytes > kRowsLdsBytes) return hipErrorInvalidValue;
  static bool allowed[kMaxDevices] = {};
  if (hipError_t status = allow_dynamic_lds(reinterpret_cast<const void *>(kernel), kRowsLdsBytes, allowed)) return status;
  constexpr uint32_t columns = DUAL ? CT * 16 : CT * 32;
  uint32_t tiles = 0;
  for (uint32_t i = 0; i < p.segments; ++i) tiles += p.tiles[i] = (p.n[i] + columns - 1) / columns;
  kernel<<<dim3(tiles, (p.m + ROWS - 1) / ROWS), CT * P * 64, bytes, stream>>>(p, norm);
  return hipGetLastError();
}

static_assert(kRowGroup == kGemvMaxRows);

uint32_t cus() { return (uint32_t)device_compute_units(); }

bool pieces_aligned(const void *x, const void *w) {
  return ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) & 15) == 0;
}

}  // namespace

bool w4a16_rows_ok(const W4LinearArgs &a) {
  return a.y_f32 == nullptr && pieces_aligned(a.x, a.w.weight) &&
         linear_rows_tile(a.m, a.n, a.k, cus()) != RowsTile::kNone;
}

hipError_t launch_w4a16_rows_linear(const W4LinearArgs &a, hipStream_t stream) {
  RowsParams p = {};
  p.x = a.x;
  p.m = a.m;
  p.k = a.k;
  p.w[0] = a.w.weight;
  p.s[0] = a.w.scale;
  p.y[0] = a.y;
  p.n[0] = a.n;
  p.segments = 1;
  p.addend = a.has_addend ? a.addend : nullptr;
  p.addend_stride = a.addend_row_stride;
  return launch_tile<false>(linear_rows_tile(a.m, a.n, a.k, cus()), p, stream);
}

bool w4a16_rows_pairs_ok(const uint16_t *x, const W4Matrix &w, uint32_t rows, uint32_t n, uint32_t k) {
  return pieces_aligned(x, w.weight) && logits_rows_tile(rows, n, k, cus()) != RowsTile::kNone;
}

hipError_t launch_w4a16_rows_pairs(const uint16_t *x, const W4Matrix &w, float *y, uint32_t rows, uint32_t n, uint32_t k,
                                   hipStream_t stream) {
  RowsParams p = {};
  p.x = x;
  p.m = rows;
  p.k = k;
  p.w[0] = w.weight;
  p.s[0] = w.scale;
  p.n[0] = n;
  p.segments = 1;
  p.pairs = y;
  return launch_tile<false>(logits_rows_tile(rows, n, k, cus()), p, stream);
}

bool w4a16_rows_ok(const W4QkvArgs &a) {
  for (int i = 0; i < 3; ++i)
    if (a.n[i] == 0 || !pieces_aligned(a.x, a.w[i].weight)) return false;
  return a.norm.weight == nullptr && qkv_rows_tile(a.m, a.n, a.k, cus()) != RowsTile::kNone;
}

hipError_t launch_w4a16_rows_qkv(const W4QkvArgs &a, hipStream_t stream) {
  RowsParams p = {};
  p.x = a.x;
  p.m = a.m;
  p.k = a.k;
  for (int i = 0; i < 3; ++i) {
    p.w[i] = a.w[i].weight;
    p.s[i] = a.w[i].scale;
    p.y[i] = a.y[i];
    p.n[i] = a.n[i];
  }
  p.segments = 3;
  return launch_tile<false>(qkv_rows_tile(a.m, a.n, a.k, cus()), p, stream);
}

bool w4a16_rows_pack_ok(const W4QkvArgs &a, const RotaryPackArgs &r) {
  return w4a16_rows_ok(a) && r.rotary.batches == 1 && r.rotary.width == 64 && pack_rows_tile(a.m, a.n, a.k, cus()) != RowsTile::kNone;
}

hipError_t launch_w4a16_rows_qkv_pack(const W4QkvArgs &a, const RotaryPackArgs &r, hipStream_t stream) {
  PackParams p = {};
  p.x = a.x;
  p.m = a.m;
  p.k = a.k;
  uint16_t *const out[3] = {r.rotary.q_output, r.rotary.k_output, a.y[2]};
  for (int i = 0; i < 3; ++i) {
    p.w[i] = a.w[i].weight;
    p.s[i] = a.w[i].scale;
    p.y[i] = out[i];
    p.n[i] = a.n[i];
  }
  p.segments = 3;
  p.cosine = r.rotary.cosine;
  p.sine = r.rotary.sine;
  p.slots = r.pack.slots;
  p.pool = r.pack.pool;
  p.token_stride = r.pack.token_stride;
  p.token_elements = r.pack.token_elements;
  for (int i = 0; i < 2; ++i) p.segment_offset[i] = r.pack.segment_offset[i];
  const RowsTile tile = pack_rows_tile(a.m, a.n, a.k, cus());
  return a.norm.weight != nullptr ? run_normed_rows<32, 2, 4, false>(p, a.norm, stream) : launch_tile<false>(tile, p, stream);
}

bool w4a16_rows_norm_ok(const W4QkvArgs &a, const W4Norm &norm, const RotaryPackArgs &r) {
  return pieces_aligned(a.x, norm.weight) && norm.weight_first == 0 && w4a16_rows_pack_ok(a, r) &&
         normed_rows(pack_rows_tile(a.m, a.n, a.k, cus()), a.m, a.n, 3, a.k, cus());
}

bool w4a16_rows_norm_ok(const W4DualSwigluArgs &a, const W4Norm &norm) {
  const uint32_t columns = 2 * a.n;
  return pieces_aligned(a.x, norm.weight) && norm.weight_first != 0 && w4a16_rows_ok(a) && a.n <= 0x7fffffffu &&
         normed_rows(gated_rows_tile(a.m, a.n, a.k, cus()), a.m, &columns, 1, a.k, cus());
}

bool w4a16_rows_ok(const W4DualSwigluArgs &a) {
  return a.norm.weight == nullptr && pieces_aligned(a.x, a.gate.weight) &&
         pieces_aligned(a.x, a.up.weight) && gated_rows_tile(a.m, a.n, a.k, cus()) != RowsTile::kNone;
}

hipError_t launch_w4a16_rows_dual_swiglu(const W4DualSwigluArgs &a, hipStream_t stream) {
  RowsParams p = {};
  p.x = a.x;
  p.m = a.m;
  p.k = a.k;
  p.w[0] = a.gate.weight;
  p.s[0] = a.gate.scale;
  p.w[1] = a.up.weight;
  p.s[1] = a.up.scale;
  p.y[0] = a.product;
  p.n[0] = a.n;
  p.segments = 1;
  const RowsTile tile = gated_rows_tile(a.m, a.n, a.k, cus());
  return a.norm.weight != nullptr ? run_normed_rows<32, 2, 4, true>(p, a.norm, stream) : launch_tile<true>(tile, p, stream);
}

}  // namespace llmopt
