"""Which tile a product takes, asked of the rules that the launches use: every tile is reached by a size that the GPU tests
run, and sizes that were measured on both sides of a line lie on the faster one (256 compute units)."""
import ctypes
import os
import subprocess

import pytest

from tests import (test_gpu_attention_tiles, test_gpu_delta_chunks, test_gpu_dense_attention, test_gpu_dense_tiles,
                   test_gpu_joined_shares, test_gpu_product_parts, test_gpu_w4a16_rows)

CUS = 256
KERNELS = os.path.join(os.path.dirname(__file__), "..", "llmopt_amd", "csrc", "kernels")
SOURCE = """
#include "chunk_join_rule.h"
#include "delta_rule.h"
#include "dense_attention_rule.h"
#include "dense_tile_rule.h"
#include "w4a16_gemm_rule.h"
#include "w4a16_rows_rule.h"
using namespace llmopt;
extern "C" {
int linear_tile(uint32_t m, uint32_t n, uint32_t k, uint32_t cus) { return (int)linear_rows_tile(m, n, k, cus); }
int gated_tile(uint32_t m, uint32_t n, uint32_t k, uint32_t cus) { return (int)gated_rows_tile(m, n, k, cus); }
int logits_tile(uint32_t tokens, uint32_t n, uint32_t k, uint32_t cus) { return (int)logits_rows_tile(2 * tokens, n, k, cus); }
int eight_waves(uint32_t causal, uint32_t rows, uint32_t keys, uint32_t past, uint32_t heads, uint32_t cus) {
  return eight_wave_slabs(64, false, causal != 0, rows, keys, past, (rows + 31) / 32 * heads, cus);
}
int turns(uint32_t dim, uint32_t masked, uint32_t causal, uint32_t rows, uint32_t keys, uint32_t past, uint32_t heads, uint32_t cus) {
  return (int)turns_form(dim, masked != 0, causal != 0, rows, keys, past, (uint64_t)((rows + 127) / 128) * heads, dim, cus);
}
int turns_of(uint32_t dim, uint32_t rows, uint32_t keys, uint64_t workgroups, uint64_t value_row_halfs, uint32_t cus) {
  return (int)turns_form(dim, false, false, rows, keys, 0, workgroups, value_row_halfs, cus);
}
uint32_t kv_head(uint32_t head, uint32_t heads, uint32_t kv_heads) { return kv_head_of(head, heads, kv_heads); }
uint32_t head_of(uint32_t rank, uint32_t heads, uint32_t kv_heads) { return turns_head(rank, heads, kv_heads); }
uint32_t walked(uint32_t any, uint32_t low, uint32_t high, uint32_t start, uint32_t every, uint32_t here) {
  const TurnsSteps steps = turns_steps(any != 0, low, high, start, every, here);
  return steps.first < steps.last ? steps.first << 16 | steps.last : 0;
}
int chunked(uint32_t dim, uint32_t capped, uint32_t m, uint32_t span, uint32_t heads) {
  return chunk_turns(dim, capped != 0, m, span, heads);
}
int three_workgroups(uint32_t tokens, uint32_t heads, uint32_t cus) {
  return three_delta_workgroups((tokens + 63) / 64 * heads, cus);
}
int large_tile(uint32_t m, uint32_t n, uint32_t k, uint32_t cus) { return (int)w4_gemm_tile(m, n, k, cus); }
int large_pair_tile(uint32_t m, uint32_t n, uint32_t k, uint32_t cus) { return (int)w4_gemm_pair_tile(m, n, k, cus); }
int product_tile(uint32_t m, uint32_t n, uint32_t k, uint32_t cus) { return (int)dense_tile(m, n, k, cus); }
int staggered_tile(uint32_t m, uint32_t n, uint32_t k, uint32_t cus) { return (int)dense_product_tile(m, n, k, cus); }
int split_columns(uint32_t m, uint32_t n, uint32_t k, uint32_t cus) { return (int)dense_first_columns(m, n, k, cus); }
float split_share(uint32_t m, uint32_t n, uint32_t k, uint32_t cus) {
  const uint64_t first = dense_first_columns(m, n, k, cus);
  float one = 0.0f, rest = 0.0f;
  dense_product_tile(m, n, k, cus, &one);
  dense_product_tile(m, n - first, k, cus, &rest);
  return (staggered_time(kStaggeredTimes[0], (uint64_t)((m + 255) / 256) * (first / 256), n, k, cus) + rest) / one;
}
float step_estimate(uint32_t m, uint32_t n, uint32_t k, uint32_t cus) {
  float time = 0.0f;
  dense_tile(m, n, k, cus, &time);
  return time;
}
float product_estimate(uint32_t m, uint32_t n, uint32_t k, uint32_t cus) {
  float time = 0.0f;
  dense_product_tile(m, n, k, cus, &time);
  return time;
}
int product_parts(uint32_t m, uint32_t n, uint32_t k, uint32_t pair, uint32_t cus) {
  const uint64_t columns = (uint64_t)n * (pair ? 2 : 1);
  if (dense_first_columns(m, columns, k, cus) != 0) return 0;
  return (int)dense_parts(dense_product_tile(m, columns, k, cus), m, columns, k, pair != 0, cus);
}
int joined(uint32_t capacity, uint32_t heads, uint32_t kv_heads, uint32_t vdim, uint32_t counters) {
  return joins((capacity + 127) / 128, heads, kv_heads, vdim, counters, 3200);
}
int normed_pair(uint32_t m, uint32_t n, uint32_t k, uint32_t cus) {
  const uint32_t columns = 2 * n;
  return normed_rows(gated_rows_tile(m, n, k, cus), m, &columns, 1, k, cus);
}
int normed_qkv(uint32_t m, uint32_t q, uint32_t kv, uint32_t k, uint32_t cus) {
  const uint32_t n[3] = {q, kv, kv};
  return normed_rows(pack_rows_tile(m, n, k, cus), m, n, 3, k, cus);
}
int qkv_tile(uint32_t m, uint32_t q, uint32_t kv, uint32_t k, uint32_t cus) {
  const uint32_t n[3] = {q, kv, kv};
  return (int)qkv_rows_tile(m, n, k, cus);
}
}
"""
DENSE = ("256x256", "128x128", "192x128", "128x192", "192x128 eight waves", "128x128 eight waves", "64x128 eight waves", "64x64",
         "32x64", "64x128")
LARGE = ("128x128", "128x128 deep", "256x128", "128x256", "256x256")
NONE, K32X32, K32X64, K32X64_DEEP, K32X64_LONG, K64X64, K64X128 = range(7)


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    folder = tmp_path_factory.mktemp("rules")
    (folder / "rules.cpp").write_text(SOURCE)
    library = str(folder / "rules.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I", KERNELS, str(folder / "rules.cpp"),
                    "-o", library], check=True)
    loaded = ctypes.CDLL(library)
    for estimate in (loaded.split_share, loaded.step_estimate, loaded.product_estimate):
        estimate.restype = ctypes.c_float
    return loaded


def sizes(test, names):
    """The sizes that a GPU test is run at."""
    return next(mark.args[1] for mark in test.pytestmark if mark.name == "parametrize" and mark.args[0] == names)


def test_gpu_tests_reach_every_tile(rules):
    tests = test_gpu_w4a16_rows
    assert {rules.linear_tile(m, n, k, CUS) for m, n, k in sizes(tests.test_small_tiles, "m,n,k")} >= set(range(1, 7))
    assert {rules.gated_tile(m, n, k, CUS) for m, n, k in sizes(tests.test_small_pair_tiles, "m,n,k")} >= set(range(2, 7))
    three = sizes(tests.test_small_tiles_over_three_matrices, "m,k,sizes")
    assert {rules.qkv_tile(m, n[0], n[1], k, CUS) for m, k, n in three} >= {K32X32, K32X64, K32X64_DEEP, K64X128}
    heads = {rules.logits_tile(m, n, k, CUS) for m, n, k in sizes(tests.test_logits_of_several_rows, "m,n,k")}
    assert heads >= {NONE, K32X32, K32X64, K64X128}


def test_96_rows_where_they_are_one_round_and_64_are_not(rules):
    tests, tall = test_gpu_w4a16_rows, K64X128 + 1
    assert {rules.linear_tile(m, n, k, CUS) for m, n, k in tests.TALL} == {tall}
    assert {rules.gated_tile(m, n, k, CUS) for m, n, k in tests.TALL_PAIRS} == {tall}
    assert rules.qkv_tile(700, 2048, 512, 576, CUS) == rules.qkv_tile(705, 1920, 640, 64, CUS) == tall
    # one round of 64 rows; more than one of 96; as many tiles of either
    assert rules.linear_tile(640, 3200, 576, CUS) == rules.gated_tile(640, 1536, 576, CUS) == K64X128
    assert rules.linear_tile(1000, 3072, 576, CUS) == NONE and rules.gated_tile(1000, 1536, 576, CUS) == K64X128
    assert rules.linear_tile(128, 17000, 1600, CUS) == K64X128


@pytest.mark.parametrize("m,k,n", [(64, 1024, 1024), (32, 2048, 2048), (64, 4096, 1024), (16, 2048, 4096), (80, 3072, 768),
                                   (40, 1536, 1536), (128, 4096, 512), (40, 1280, 1280)])
def test_few_row_groups(rules, m, k, n):
    """Up to two groups a CU the GEMV is the faster one, beyond that a tile is."""
    assert rules.linear_tile(m, n, k, CUS) == NONE
    assert rules.linear_tile(m + 24, n, k, CUS) != NONE or m + 24 > 128
    assert rules.linear_tile(m + 24, n + 512, k, CUS) != NONE


@pytest.mark.parametrize("m,k,n", [(64, 1024, 1024), (32, 2048, 2048), (56, 1536, 576), (64, 4096, 1024), (128, 2048, 512),
                                   (16, 1024, 4096), (40, 768, 768), (128, 1024, 512), (112, 4096, 256)])
def test_few_row_groups_of_pairs(rules, m, k, n):
    assert rules.gated_tile(m, n, k, CUS) == NONE


@pytest.mark.parametrize("m,k,n", [(72, 1024, 1024), (40, 2048, 2048), (72, 4096, 1024), (128, 1536, 576), (64, 512, 1024),
                                   (33, 512, 2048), (16, 2048, 4096)])
def test_pairs_beyond_the_row_groups(rules, m, k, n):
    assert rules.gated_tile(m, n, k, CUS) != NONE


@pytest.mark.parametrize("tokens,k,n,tiles", [
    (8, 2048, 32000, False), (12, 2048, 32000, False), (8, 3072, 32000, False), (8, 4096, 16384, False), (12, 4096, 32000, False),
    (8, 8192, 8192, False), (16, 2048, 2048, False), (5, 2048, 16384, False), (4, 2048, 32000, False),
    (5, 576, 49152, True), (32, 576, 49152, True), (12, 1536, 32000, True), (12, 2048, 16384, True), (16, 2048, 32000, True),
    (12, 4096, 16384, True), (20, 4096, 32000, True), (64, 4096, 32000, True), (16, 8192, 8192, True), (20, 4096, 8192, True)])
def test_logits(rules, tokens, k, n, tiles):
    """Few rows and a long K stay with the GEMV also where 64 x 128 tiles would be one round."""
    assert (rules.logits_tile(tokens, n, k, CUS) != NONE) == tiles


@pytest.mark.parametrize("causal,rows,keys,past,heads,eight", [
    (1, 700, 700, 0, 9, 1), (1, 900, 900, 0, 9, 1), (1, 64, 2000, 1936, 9, 1), (1, 400, 4000, 3600, 9, 1), (0, 32, 4096, 0, 9, 1),
    (1, 1000, 1000, 0, 9, 1), (0, 512, 560, 0, 16, 1), (1, 512, 1024, 512, 16, 1),
    # a second round
    (0, 560, 560, 0, 16, 0), (1, 560, 560, 0, 16, 0), (0, 1000, 1000, 0, 9, 0), (1, 1025, 1025, 0, 9, 0),
    (1, 512, 512, 0, 9, 0), (1, 700, 700, 0, 32, 0), (1, 2048, 2048, 0, 9, 0),
    # keys beyond the causal limit of the last row are not walked
    (1, 32, 4096, 0, 9, 0), (1, 64, 2000, 0, 16, 0), (1, 100, 520, 0, 3, 0), (1, 32, 4096, 224, 9, 0), (1, 32, 4096, 225, 9, 1), (1, 400, 4000, 0, 9, 1)])
def test_eight_waves_a_slab(rules, causal, rows, keys, past, heads, eight):
    assert rules.eight_waves(causal, rows, keys, past, heads, CUS) == eight


@pytest.mark.parametrize("heads,kv_heads", [(9, 3), (32, 32), (7, 1), (131072, 65536), (100000, 50000), (131070, 43690),
                                            (1 << 31, 1 << 30), (0xfffffffe, 0x7fffffff)])
def test_key_head_of_a_query_head(rules, heads, kv_heads):
    """Also where heads times kv_heads is more than 32 bits hold."""
    rules.kv_head.restype = ctypes.c_uint32
    for head in {0, 1, heads // kv_heads, heads // 3, heads // 2, heads - 2, heads - 1}:
        assert rules.kv_head(ctypes.c_uint32(head), ctypes.c_uint32(heads), ctypes.c_uint32(kv_heads)) == head * kv_heads // heads


@pytest.mark.parametrize("dim,masked,rows,keys,heads,form", [
    (128, 0, 4096, 4096, 32, 2), (128, 0, 3500, 3500, 32, 2), (128, 0, 3000, 3000, 32, 1), (128, 0, 1000, 9000, 128, 1),
    (128, 0, 300, 300, 32, 0), (128, 0, 700, 700, 32, 1), (128, 0, 1000, 1000, 16, 0), (128, 0, 1100, 1100, 16, 1),
    (128, 0, 255, 255, 80, 0), (128, 0, 255, 256, 80, 1), (64, 0, 2040, 2040, 16, 1), (64, 0, 1900, 1900, 16, 0), (64, 0, 4096, 4096, 32, 2),
    (256, 0, 4096, 4096, 32, 0), (128, 0, 300, 300, 512, 0), (128, 0, 300, 800, 256, 1), (128, 0, 64, 1000, 1024, 1), (128, 1, 4096, 4096, 32, 0)])
def test_attention_in_turns(rules, dim, masked, rows, keys, heads, form):
    assert rules.turns(dim, masked, 0, rows, keys, 0, heads, CUS) == form


@pytest.mark.parametrize("dim,causal,rows,past,heads,form", [
    (128, 1, 520, 0, 30 * 16, 0), (128, 1, 520, 0, 6 * 16, 1), (128, 1, 700, 0, 20 * 16, 0), (64, 1, 520, 0, 16 * 9, 0), (64, 1, 924, 0, 10 * 9, 0),
    (64, 1, 300, 0, 52 * 9, 0), (128, 0, 300, 0, 256, 0), (128, 0, 64, 448, 1024, 0), (128, 0, 128, 472, 75 * 32, 0), (128, 0, 128, 872, 75 * 32, 1),
    (128, 1, 520, 280, 4 * 32, 0), (128, 1, 1000, 300, 3 * 32, 1), (128, 1, 924, 600, 7 * 16, 1), (64, 1, 700, 600, 7 * 16, 1),
    (128, 1, 1030, 0, 17 * 16, 2), (64, 1, 1100, 0, 24 * 16, 2), (64, 1, 1030, 0, 9 * 9, 1), (128, 1, 1030, 0, 4 * 16, 0),
    (128, 1, 16, 0xfffffff0, 800, 1)])
def test_long_walks_of_many_workgroups_go_in_turns(rules, dim, causal, rows, past, heads, form):
    """More than two workgroups a CU: what a workgroup walks on average decides."""
    assert rules.turns(dim, 0, causal, rows, min(past + rows, 2000), past if causal else 0, heads, CUS) == form


def turns_offsets(dim, waves, values, stride_bytes):
    """TurnsCopy::offset (attention_turns.h) of every copy and thread: where it reads behind the stage's first row, less what the
    instruction's own offset adds."""
    pieces = dim // 8
    keys = 64 // pieces
    count = 64 // keys // waves
    for c in range(count):
        for thread in range(64 * waves):
            row = (thread // 64 % waves * count + c) * keys + thread % 64 // pieces
            piece = (thread % pieces) ^ ((2 if values else 1) * row & (pieces - 1))
            yield row * stride_bytes + piece * 16 - c * 1024


@pytest.mark.parametrize("dim", [64, 128])
def test_value_rows_of_turns_in_32_bits(rules, dim):
    """Token-first values of many key heads: the longest rows that go in turns have all their places in 32 bits; longer ones,
    from 262144 heads of 128 on, keep the tiles of 64-bit addresses."""
    form = lambda halfs: rules.turns_of(dim, 128, 2000, ctypes.c_uint64(halfs // dim), ctypes.c_uint64(halfs), CUS)
    longest = (1 << 25) - dim
    assert form(longest) != 0
    for waves in (4, 8):
        for values in (False, True):
            for stride in (dim, longest):
                offsets = list(turns_offsets(dim, waves, values, stride * 2))
                assert min(offsets) >= 0 and max(offsets) < 1 << 32
    for halfs in (1 << 25, 266306 * 128, 1 << 31, 1 << 33):
        assert form(halfs) == 0


@pytest.mark.parametrize("heads,kv_heads", [(32, 8), (16, 4), (9, 3), (7, 7), (130, 13), (60, 20), (3000, 750), (640, 64)])
def test_order_of_heads_in_turns(rules, heads, kv_heads):
    """Every head once; those of a key head close together, on one XCD of eight if key heads come in whole eights."""
    order = [rules.head_of(rank, heads, kv_heads) for rank in range(heads)]
    assert sorted(order) == list(range(heads))
    per = heads // kv_heads
    ranks = [sorted(rank for rank, head in enumerate(order) if head // per == kv) for kv in range(kv_heads)]
    assert all(r[-1] - r[0] <= 8 * (per - 1) for r in ranks)
    assert kv_heads % 8 != 0 or all(len({rank % 8 for rank in r}) == 1 for r in ranks)


@pytest.mark.parametrize("every", [1, 2])
def test_steps_that_a_wave_of_rows_walks(rules, every):
    """The steps whose 64 keys hold any that the wave's rows see, and none for a wave whose rows lie past the end."""
    for start in (0, 64, 100, 1437):
        for here in (0, 1, 2, 9):
            for low in (0, 1, 63, 64, 100, 127, 128, 129, 164, 1436, 1500, 1501, 1629):
                for high in (low + 31, low + 100, low + 700):
                    seen = [s for s in range(here) if start + s * every * 64 <= high and start + s * every * 64 + 63 >= low]
                    assert rules.walked(1, low, high, start, every, here) == (seen[0] << 16 | seen[-1] + 1 if seen else 0)
                    assert rules.walked(0, low, high, start, every, here) == 0


@pytest.mark.parametrize("dim,rows,keys", [(64, 16, 1500), (128, 128, 4096), (64, 1024, 1024)])
def test_turns_keep_to_grids_of_fewer_than_32_bits_of_threads(rules, dim, rows, keys):
    """2^23 workgroups of 512 threads are more than a launch takes; 256-thread workgroups are not."""
    form = lambda workgroups: rules.turns_of(dim, rows, keys, ctypes.c_uint64(workgroups), ctypes.c_uint64(dim), CUS)
    assert form((1 << 23) - 1) != 0
    assert form(1 << 23) == form((1 << 24) - 1) == form((1 << 31) - 1) == 0
    assert rules.chunked(dim, 0, 1025, 4096, ((1 << 23) - 1) // 9) == 1
    assert rules.chunked(dim, 0, 1025, 4096, (1 << 23) // 9 + 1) == 0


def test_gpu_tests_reach_both_forms_of_turns(rules):
    names = "dim,batches,heads,kv_heads,new,past,mode"
    reached = [(dim, rules.turns(dim, 0, int(mode == "causal"), new, new + past, past, heads * batches, CUS))
               for dim, batches, heads, _, new, past, mode in sizes(test_gpu_dense_attention.test_groups_of_waves_in_turns, names)]
    assert set(reached) == {(64, 1), (64, 2), (128, 1), (128, 2)}
    for dim, heads, _, new, past in sizes(test_gpu_dense_attention.test_rows_that_see_one_stage_of_many, "dim,heads,kv_heads,new,past"):
        assert rules.turns(dim, 0, 1, new, new + past + 300, past, heads, CUS) == 1


@pytest.mark.parametrize("dim,capped,m,span,turns", [
    (128, 0, 3001, 2048, 1), (128, 0, 513, 0, 1), (128, 0, 1500, 512, 0), (128, 0, 500, 2048, 0), (128, 1, 2048, 2048, 1),
    (128, 1, 3001, 1024, 1), (128, 1, 1000, 2048, 0), (128, 1, 2000, 512, 0), (64, 0, 1500, 2048, 1), (64, 0, 3001, 1024, 0),
    (64, 1, 3001, 2048, 0), (96, 0, 3001, 2048, 0), (256, 0, 3001, 2048, 0)])
def test_portions_in_turns(rules, dim, capped, m, span, turns):
    assert rules.chunked(dim, capped, m, span, 16) == turns


def test_gpu_tests_of_portions_go_in_turns(rules):
    for m, heads, _, dim, _, span, softcap, *_ in sizes(test_gpu_attention_tiles.test_groups_of_waves_in_turns,
                                                    "m,heads,kv,dim,vdim,span,softcap,sink,first,sliding"):
        assert rules.chunked(dim, int(softcap > 0), m, span, heads) == 1


@pytest.mark.parametrize("tokens,heads,three", [(3001, 16, 1), (2115, 16, 1), (4096, 32, 1), (3001, 32, 1), (3001, 8, 0),
                                                (2048, 16, 0), (4096, 16, 0), (1000, 64, 0), (100, 4, 0)])
def test_three_workgroups_of_the_delta_rule(rules, tokens, heads, three):
    """Where they save a round, and only there."""
    assert rules.three_workgroups(tokens, heads, CUS) == three


def test_gpu_tests_reach_three_workgroups(rules):
    names = "m,heads,kv_heads,dim,vdim"
    for m, heads, _, dim, _ in sizes(test_gpu_delta_chunks.test_three_workgroups_against_float64, names):
        assert 64 < dim <= 128 and rules.three_workgroups(m, heads, CUS) == 1


def test_gpu_tests_reach_every_product_tile(rules):
    tests, every = test_gpu_dense_tiles, set(range(len(DENSE)))
    assert {rules.product_tile(*size, CUS) for size in sizes(tests.test_tiles, "m,n,k")} == every
    assert {rules.product_tile(m, 2 * ff, width, CUS) for m, width, ff in sizes(tests.test_gated_tiles, "m,width,ff")} == every
    assert {rules.product_tile(*size, CUS) for size in tests.ROW_SIZES} == every


@pytest.mark.parametrize("m,n,k,tile", [
    (1500, 2048, 128, "64x128"), (3001, 1024, 256, "64x128"), (700, 4096, 128, "64x128"), (64, 4096, 128, "32x64"),
    (700, 4096, 512, "128x128 eight waves"), (2048, 2048, 4096, "128x128 eight waves"), (512, 6144, 2048, "128x128 eight waves"),
    (3001, 2048, 128, "192x128 eight waves"), (3001, 2048, 4096, "192x128 eight waves"), (2048, 6144, 2048, "128x192"),
    (300, 12288, 512, "64x128"), (384, 2816, 8192, "64x64"), (700, 5632, 2048, "64x128"), (900, 8192, 1024, "128x128"),
    (2048, 9504, 1024, "192x128"), (2048, 12288, 512, "128x192"), (700, 1500, 8192, "64x64"), (3001, 9504, 2048, "256x256"),
    (512, 2048, 4096, "64x64"), (64, 4384, 1024, "32x64"), (3001, 8192, 2048, "192x128"), (2048, 4224, 2048, "192x128"),
    (1024, 2048, 4096, "64x128 eight waves")])
def test_product_tiles(rules, m, n, k, tile):
    """The least of the ten estimates: what a product runs on below K = 1024, and what the staggered tiles are held against."""
    assert DENSE[rules.product_tile(m, n, k, CUS)] == tile


def test_gpu_tests_reach_every_staggered_tile(rules):
    every = {DENSE.index("256x256")} | set(range(len(DENSE), len(DENSE) + 5))
    assert {rules.staggered_tile(*size, CUS) for size in test_gpu_dense_tiles.STAGGERED} == every
    assert {rules.staggered_tile(m, n // 2 * 2, k, CUS) for m, n, k in test_gpu_dense_tiles.STAGGERED} == every
    assert all(0 < rules.split_columns(m, n // 2 * 2, k, CUS) < n for m, n, k in test_gpu_dense_tiles.SPLIT)


@pytest.mark.parametrize("m,n,k", [(2048, 2048, 1000), (64, 4096, 1024), (3001, 2048, 128), (2048, 2048, 512), (330, 700, 2048)])
def test_products_that_stay_in_step(rules, m, n, k):
    """A short K, and launches that no staggered tile fills."""
    assert rules.staggered_tile(m, n, k, CUS) == rules.product_tile(m, n, k, CUS)


@pytest.mark.parametrize("m,n,k", [(223, 10624, 1408), (751, 5312, 1408), (220, 9984, 1600), (213, 14656, 1408), *test_gpu_dense_tiles.SHORT])
def test_128_rows_and_columns_stay_in_step_below_1792(rules, m, n, k):
    assert DENSE[rules.staggered_tile(m, n, k, CUS)] == "128x128 eight waves"
    assert rules.staggered_tile(m, n, 1792, CUS) == len(DENSE) + 1


@pytest.mark.parametrize("m,n,k,first", [(2048, 8512, 2048, 8192), (3001, 7312, 2048, 5376), (2048, 9504, 2048, 8192),
                                         (2048, 16384, 2048, 0), (3001, 16384, 2048, 0), (2048, 2048, 8192, 0), (2048, 8512, 960, 0)])
def test_columns_in_two_launches(rules, m, n, k, first):
    assert rules.split_columns(m, n, k, CUS) == first


def test_a_product_in_two_launches_is_estimated_5_percent_shorter(rules):
    """On one scale: a tile in step counts for 0.93 of its estimate, alone, as the rest and as the one launch."""
    found = 0
    for m in (700, 1171, 1422, 2048, 2701, 3001):
        for n in range(1024, 16384, 449):
            for k in (960, 1024, 1280, 2048, 3520, 8192):
                first = rules.split_columns(m, n, k, CUS)
                if rules.staggered_tile(m, n, k, CUS) == rules.product_tile(m, n, k, CUS) != DENSE.index("256x256"):
                    assert rules.product_estimate(m, n, k, CUS) == pytest.approx(0.93 * rules.step_estimate(m, n, k, CUS), rel=1e-6)
                if first:
                    found += 1
                    assert k >= 1024 and first % 256 == 0 and 0 < first < n and rules.split_share(m, n, k, CUS) < 0.95
                    assert (m + 255) // 256 * (first // 256) <= CUS * ((m + 255) // 256 * ((n + 255) // 256) // CUS)
    assert found > 100


@pytest.mark.parametrize("m,n,k", [(897, 11657, 1024), (1223, 9265, 1408), (2535, 3665, 2688), (1412, 6260, 1024)])
def test_columns_that_are_no_whole_pieces(rules, m, n, k):
    """256 x 256 tiles store them more slowly than the others do: not these sizes, which whole pieces give to them."""
    assert DENSE[rules.staggered_tile(m, n // 8 * 8, k, CUS)] == "256x256"
    assert rules.staggered_tile(m, n, k, CUS) == rules.product_tile(m, n, k, CUS)
    assert all(DENSE[rules.staggered_tile(*size, CUS)] == "192x128" for size in test_gpu_dense_tiles.ODD)


def test_rows_normalised_in_the_tile(rules):
    """Tiles of 32 rows in one round, and a whole K in LDS."""
    assert all(rules.normed_pair(m, n, k, CUS) for m, n, k in test_gpu_w4a16_rows.NORMED_PAIRS)
    assert rules.normed_qkv(700, 576, 192, 576, CUS) and rules.normed_qkv(90, 576, 192, 576, CUS)
    assert not rules.normed_pair(700, 1536, 576, CUS)       # 96 rows
    assert not rules.normed_pair(100, 1000, 832, CUS)       # thirteen groups
    assert not rules.normed_qkv(1300, 576, 192, 576, CUS)   # a second round


def test_gpu_tests_reach_the_256_tiles_of_w4a16(rules):
    """Products and pairs that the small tiles and the GEMV's row groups leave alone, by more than a round of the middle tiles."""
    tests = test_gpu_w4a16_rows
    for m, n, k, _ in sizes(tests.test_tiles_of_256, "m,n,k,addend"):
        assert rules.linear_tile(m, n, k, CUS) == NONE and LARGE[rules.large_tile(m, n, k, CUS)] == "256x256", (m, n, k)
    for m, n, k, _ in sizes(tests.test_tiles_of_128_by_256, "m,n,k,addend"):
        assert rules.linear_tile(m, n, k, CUS) == NONE and LARGE[rules.large_tile(m, n, k, CUS)] == "128x256", (m, n, k)
    for m, n, k in sizes(tests.test_pair_tiles_of_256, "m,n,k"):
        assert rules.gated_tile(m, n, k, CUS) == NONE and LARGE[rules.large_pair_tile(m, n, k, CUS)] == "256x256", (m, n, k)


@pytest.mark.parametrize("m,n,k,tile", [(2048, 14336, 4096, "256x256"), (2048, 6144, 2048, "256x256"), (1430, 5632, 576, "256x256"),
                                        (1134, 6720, 2112, "128x256"), (541, 11840, 576, "128x256"), (512, 14336, 4096, "256x128"),
                                        (2048, 4096, 4096, "256x128"), (512, 4096, 4096, "128x128 deep"),
                                        (1600, 3000, 576, "128x128"), (2048, 14336, 1 << 23, "256x128")])
def test_large_w4a16_tiles(rules, m, n, k, tile):
    assert LARGE[rules.large_tile(m, n, k, CUS)] == tile


@pytest.mark.parametrize("m,n,k,tile", [(2048, 1536, 576, "128x128 deep"), (2048, 14336, 4096, "256x256"), (2049, 2048, 576, "256x256"),
                                        (2048, 2048, 576, "128x128 deep"), (2048, 14336, 1 << 23, "128x128 deep")])
def test_large_w4a16_pair_tiles(rules, m, n, k, tile):
    assert LARGE[rules.large_pair_tile(m, n, k, CUS)] == tile


PARTS = ("none", "16x32", "32x32", "32x64")


def test_gpu_tests_reach_every_product_in_parts(rules):
    tests = test_gpu_product_parts.SIZES
    assert {PARTS[rules.product_parts(m, n, k, 0, CUS)] for m, n, k in tests} == set(PARTS)
    assert {PARTS[rules.product_parts(m, n + 40, k, 0, CUS)] for m, n, k in tests} == set(PARTS)
    assert {PARTS[rules.product_parts(m, max(16, n // 2), k, 1, CUS)] for m, n, k in tests} == {"none", "32x64"}


@pytest.mark.parametrize("m,n,k,pair,form", [
    (64, 1024, 4096, 0, "16x32"), (64, 1024, 256, 0, "16x32"), (64, 1024, 192, 0, "none"),    # a tile a CU, K = 256
    (64, 2048, 256, 0, "16x32"), (64, 2049, 256, 0, "32x32"), (64, 4096, 512, 0, "32x32"),    # 256 tiles of 16 x 32, of 32 x 32
    (64, 4097, 1024, 0, "32x64"), (64, 4097, 960, 0, "none"), (64, 8192, 1024, 0, "32x64"),   # of 32 x 64, K = 1024
    (64, 8193, 1024, 0, "none"), (500, 1024, 1024, 0, "32x64"),
    (64, 512, 1024, 1, "32x64"), (64, 512, 960, 1, "none"),                                   # a pair: a quarter of the CUs
    (16, 4096, 1024, 1, "none"), (16, 4096, 2048, 1, "32x64"),
])
def test_products_in_parts(rules, m, n, k, pair, form):
    assert PARTS[rules.product_parts(m, n, k, pair, CUS)] == form


def test_gpu_tests_reach_both_ends_of_the_join(rules):
    tests = test_gpu_joined_shares.test_shares_of_a_token
    shapes, rings = sizes(tests, "heads,kv_heads,dim,vdim"), sizes(tests, "capacity")
    for per_ring in ([rules.joined(ring, heads, kv, vdim, 1024) for ring in rings] for heads, kv, _, vdim in shapes):
        assert not per_ring[0] and not per_ring[-1]  # one share, more than 64
    assert len({tuple(rules.joined(ring, heads, kv, vdim, 1024) for ring in rings) for heads, kv, _, vdim in shapes}) >= 3


@pytest.mark.parametrize("heads,kv_heads,vdim,capacity,join", [
    (16, 4, 64, 256, 1), (16, 4, 64, 8192, 1), (16, 4, 64, 8193, 0), (16, 4, 64, 128, 0),     # 256 outputs: up to 64 shares
    (32, 8, 128, 2048, 1), (32, 8, 128, 2049, 0), (64, 4, 64, 256, 0),                        # 512: up to 16; 1024: never
    (96, 1, 5, 2048, 1), (97, 1, 5, 2048, 0),                                                 # what a workgroup's memory holds
])
def test_joined_shares(rules, heads, kv_heads, vdim, capacity, join):
    assert rules.joined(capacity, heads, kv_heads, vdim, kv_heads) == join
    assert rules.joined(capacity, heads, kv_heads, vdim, kv_heads - 1) == 0  # too few counters
