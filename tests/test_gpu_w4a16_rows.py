"""The small tiles of w4a16_rows.hip against float64 products of the oracle's dequantised weights: every tile its rule can
choose, at sizes that leave remainders of rows, columns and K steps.  The kernel keeps the nibbles exact and sums in
float32, so its error is the output's rounding: half a unit in the last place, 2^-11 relative at most (the tolerance
of the other linears, 1e-3, is twice that)."""
import struct

import numpy as np
import pytest

import oracle
from tests.gpu_util import assert_close_to_oracle, linear_grid, u32s, w4_case
from tests.test_gpu_glue import check_tokens, lm_head_oracle, run_lm_head
from tests.test_gpu_w4a16 import run_linear

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def runtime():
    from llmopt_amd.native import Runtime
    rt = Runtime()
    yield rt
    rt.close()


def product(x, packed, scale):
    return x.astype(np.float64) @ oracle.w4_dequant(packed, scale).astype(np.float64).T


# 32 x 32: one round of workgroups; 32 x 64 with a short K, with a K that fits its deep ring, with a longer one;
# 64 x 64; 64 x 128 with long and with short K
@pytest.mark.parametrize("m,n,k", [
    (129, 33, 64), (9, 5500, 1088), (70, 1000, 1088), (17, 1000, 14400), (24, 4096, 4096),
    (300, 1001, 832), (600, 700, 64), (700, 576, 576),
    (33, 4129, 1536), (33, 4100, 4096), (33, 4129, 4160), (130, 3000, 8256),
    (200, 2601, 1600), (193, 2600, 6144), (520, 2001, 1536), (1100, 1000, 576)])
@pytest.mark.parametrize("addend", ["none", "bias", "residual"])
def test_small_tiles(runtime, m, n, k, addend):
    rng = np.random.default_rng(m * 7919 + n * 31 + k)
    x, packed, scale, bias = w4_case(rng, m, n, k, bias=True)
    expected = product(x, packed, scale)
    if addend == "none":
        out = run_linear(runtime, x, packed, scale)
    elif addend == "bias":
        out, expected = run_linear(runtime, x, packed, scale, bias=bias), expected + bias.astype(np.float64)
    else:
        residual = rng.standard_normal((m, n)).astype(np.float16)
        out, expected = run_linear(runtime, x, packed, scale, residual=residual), expected + residual.astype(np.float64)
    assert_close_to_oracle(out, expected, f"linear {m}x{n}x{k} {addend}")


def test_exact_integers_and_infinities(runtime):
    """Whole-number activations and a scale of one give the product itself; an infinity stays in its row."""
    m, n, k = 129, 257, 320
    rng = np.random.default_rng(1)
    x, packed, _, _ = w4_case(rng, m, n, k)
    x = rng.integers(-4, 5, (m, k)).astype(np.float16)
    scale = np.ones((n, k // 64), dtype=np.float16)
    expected = product(x, packed, scale)
    np.testing.assert_array_equal(run_linear(runtime, x, packed, scale), expected.astype(np.float16))
    x[5, 319] = np.inf
    out = run_linear(runtime, x, packed, scale)
    assert not np.isfinite(out[5]).any()
    rows = np.arange(m) != 5
    np.testing.assert_array_equal(out[rows], expected.astype(np.float16)[rows])


@pytest.mark.parametrize("m,n,k", [
    (300, 200, 64), (100, 1537, 576), (300, 1536, 576), (600, 1000, 576), (700, 1536, 576),
    (70, 1601, 1600), (33, 2000, 4096), (65, 1000, 8256), (24, 2000, 14400), (40, 8192, 1536), (24, 14336, 1600),
    (500, 1999, 1600)])
def test_small_pair_tiles(runtime, m, n, k):
    rng = np.random.default_rng(m * 104729 + n * 13 + k)
    x, gate, gate_scale, _ = w4_case(rng, m, n, k)
    _, up, up_scale, _ = w4_case(rng, 1, n, k)
    out = runtime.buffer_of_bytes(np.full((m, n), np.nan, dtype=np.float16))
    runtime.dispatch("llmopt_w4a16_dual_swiglu_f16_g64_m4",
                     [runtime.buffer_of_bytes(a) for a in (x, gate, gate_scale, up, up_scale)] + [out],
                     u32s(m, n, k) + struct.pack("<f", 1e-5), grid=(linear_grid(((m + 3) // 4) * n), 1, 1), group=(256, 1, 1))
    g = product(x, gate, gate_scale)
    assert_close_to_oracle(out.numpy(np.float16, (m, n)), g / (1.0 + np.exp(-g)) * product(x, up, up_scale), f"pair {m}x{n}x{k}")


@pytest.mark.parametrize("m,k,sizes", [(129, 64, (64, 33, 1)), (700, 576, (576, 192, 192)), (300, 832, (577, 191, 193)),
                                       (200, 1600, (1024, 256, 257)), (40, 2048, (2048, 512, 512)), (520, 2048, (1024, 512, 500)),
                                       (1100, 576, (600, 200, 201))])
def test_small_tiles_over_three_matrices(runtime, m, k, sizes):
    rng = np.random.default_rng(m + k)
    x = rng.standard_normal((m, k)).astype(np.float16)
    mats = [w4_case(rng, 1, n, k)[1:3] for n in sizes]
    outs = [runtime.buffer_of_bytes(np.full((m, n), np.nan, dtype=np.float16)) for n in sizes]
    runtime.dispatch("llmopt_w4a16_qkv_linear_f16_g64_m4",
                     [runtime.buffer_of_bytes(x)] + [runtime.buffer_of_bytes(a) for pair in mats for a in pair] + outs,
                     u32s(m, k, *sizes), grid=(linear_grid(m * sum(sizes)), 1, 1), group=(256, 1, 1))
    for (packed, scale), out, n in zip(mats, outs, sizes):
        assert_close_to_oracle(out.numpy(np.float16, (m, n)), product(x, packed, scale), f"three matrices {m}x{n}x{k}")


# 96 x 128: rows and columns that end inside a tile, a last step of one group (K = 576) and of two, the longest K
TALL = [(700, 3072, 576), (575, 5201, 64), (300, 8100, 1600), (481, 4099, 4160), (289, 7900, 6144)]
TALL_PAIRS = [(700, 1536, 576), (575, 2561, 64), (300, 4033, 1600), (481, 2050, 4096)]


@pytest.mark.parametrize("m,n,k", TALL)
def test_tiles_of_96_rows(runtime, m, n, k):
    test_small_tiles(runtime, m, n, k, "residual")


@pytest.mark.parametrize("m,n,k", TALL_PAIRS)
def test_pair_tiles_of_96_rows(runtime, m, n, k):
    test_small_pair_tiles(runtime, m, n, k)


@pytest.mark.parametrize("k,heads,kv_heads,tokens", [(576, 32, 8, 700), (64, 30, 10, 705)])
def test_projection_with_rotation_and_pack_on_96_rows(runtime, k, heads, kv_heads, tokens):
    test_projection_with_rotation_and_pack(runtime, k, heads, kv_heads, 64, tokens)


# float32 logits from pairs of rows: one round of small tiles, 32 x 64 with short and with long K, 64 x 128, and the
# matrix-core GEMV on the other side of the rule (few rows, long K)
@pytest.mark.parametrize("m,n,k", [
    (30, 2047, 64), (5, 33001, 576), (16, 16387, 576), (17, 33003, 320), (130, 10001, 576), (13, 24001, 1600),
    (40, 20002, 1536), (12, 24001, 1536), (8, 16401, 2048), (12, 33001, 2112)])
@pytest.mark.parametrize("dtype", [np.float16, np.float32])
def test_logits_of_several_rows(runtime, m, n, k, dtype):
    rng = np.random.default_rng(m * 31 + n)
    x, packed, scale, _ = w4_case(rng, m, n, k)
    x, weight = x.astype(dtype), rng.uniform(0.5, 1.5, k).astype(np.float16)
    tokens, logits = run_lm_head(runtime, x, weight, packed, scale, 1e-5, extra=True)
    expected = lm_head_oracle(x, weight, packed, scale, 1e-5)
    check_tokens(tokens, expected)
    assert_close_to_oracle(logits, expected, f"logits {m}x{n}x{k}")


# width, query heads, key / value heads, tokens: two launches (few tokens: the decode projection; heads of 128), 32 x 64
# where half a head's columns would be the tile, 32 x 64, 64 x 64 and 64 x 128 tiles of whole heads, large tiles
@pytest.mark.parametrize("k,heads,kv_heads,dim,tokens", [
    (576, 9, 3, 64, 7), (576, 9, 3, 64, 40), (320, 4, 2, 128, 200), (576, 9, 3, 64, 90), (64, 3, 1, 64, 333), (576, 9, 3, 64, 700),
    (2048, 8, 2, 64, 70), (4160, 16, 8, 64, 33), (1600, 32, 8, 64, 193), (576, 32, 8, 64, 520), (576, 32, 8, 64, 2048)])
def test_projection_with_rotation_and_pack(runtime, k, heads, kv_heads, dim, tokens):
    """The entry against the two that it joins: the rotated queries and keys, the values and the pool bit for bit where
    both run the same tile, slots in any order, a key / value row of zeros (whose scale is one), bytes of other layers and tokens left alone."""
    rng = np.random.default_rng(tokens + k)
    n = (heads * dim, kv_heads * dim, kv_heads * dim)
    x, norm = rng.standard_normal((tokens, k)).astype(np.float16), rng.uniform(0.5, 1.5, k).astype(np.float16)
    x[tokens // 2] = 0
    put = runtime.buffer_of_bytes
    matrices = [put(a) for rows in n for a in w4_case(rng, 1, rows, k)[1:3]]
    angle = rng.uniform(0, 6.3, (tokens, dim // 2)).astype(np.float32)
    cosine, sine = (put(np.concatenate([f(angle)] * 2, axis=1).astype(np.float16)) for f in (np.cos, np.sin))
    elements, stride = 4 * n[1], 4 * n[1] + 4 * n[1] // 32 + 6
    slots = put(rng.permutation(tokens + 3)[:tokens].astype(np.uint32))
    pool = rng.integers(0, 256, (tokens + 3) * stride, dtype=np.uint8)
    projection = u32s(tokens, k, *n) + struct.pack("<f", 1e-5)
    pack = u32s(1, tokens, heads, kv_heads, dim, dim // 2, 1) + \
        u32s(tokens, n[1], 3 * n[1], kv_heads, dim, 64, elements, elements // 64, stride, tokens, 0)
    results = []
    for joined in (False, True):
        create = lambda i: put(np.full(tokens * n[i], np.nan, dtype=np.float16))
        q_out, k_out, v_out, b_pool = create(0), create(1), create(2), put(pool)
        if joined:
            runtime.dispatch("llmopt_rms_w4a16_qkv_rotary_pack_prompt_q8_f16_g64",
                             [put(x), put(norm), *matrices, cosine, sine, q_out, k_out, v_out, slots, b_pool],
                             projection + pack, (linear_grid(sum(n)), 1, 1), (256, 1, 1))
        else:
            q, k_raw = create(0), create(1)
            runtime.dispatch("llmopt_rms_w4a16_qkv_linear_f16_g64", [put(x), put(norm), *matrices, q, k_raw, v_out],
                             projection, (linear_grid(sum(n)), 1, 1), (256, 1, 1))
            runtime.dispatch("llmopt_rotary_qk_pack_q8_batched",
                             [q, k_raw, cosine, sine, q_out, k_out, v_out, slots, b_pool], pack, (256, 1, 1), (256, 1, 1))
        results.append([b.numpy(np.uint8) for b in (q_out, k_out, v_out, b_pool)])
    if (k, tokens) in ((576, 90), (4160, 33)):
        # the projection alone takes the tile of half a head's columns, whose sums add in another order: a value moves by
        # one rounding to half (2^-10 of itself) at most and takes two of them and their products' roundings along, a
        # scale by as many units in its last place, a quantised value by one step
        for two, one in zip(*(r[:3] for r in results)):
            two, one = two.view(np.float16).astype(np.float32), one.view(np.float16).astype(np.float32)
            assert np.abs(one - two).max() <= 4 * 2.0 ** -10 * np.abs(two).max()
        two, one = (r[3].reshape(-1, stride) for r in results)
        scales = slice(elements, elements + elements // 32)
        for a, b, steps in ((one[:, :elements].view(np.int8), two[:, :elements].view(np.int8), 1),
                            (np.ascontiguousarray(one[:, scales]).view(np.uint16),
                             np.ascontiguousarray(two[:, scales]).view(np.uint16), 4)):
            assert np.abs(a.astype(np.int32) - b.astype(np.int32)).max() <= steps
        return
    for name, two, one in zip(("queries", "keys", "values", "pool"), *results):
        np.testing.assert_array_equal(one, two, err_msg=name)
    assert np.isfinite(results[1][0].view(np.float16)).all()


def test_logits_of_more_rows_than_a_grid_of_tiles_has():
    """A hi and a lo row each of 32 * 65536 tokens and some: every token's logits against float64.  They are rounded to
    half, 2^-11 of the value; the GEMV's weights are nibbles with a bias of up to 1032, which a second sum takes out
    again: 64 additions of 2^-24 of sums up to 1040 times those of the activations each."""
    from llmopt_amd.native import Runtime
    runtime = Runtime()
    m, n, k = 32 * 65536 + 40, 5, 64
    g = torch.Generator(device="cuda").manual_seed(6)
    x = torch.randn(m, k, generator=g, device="cuda").half()
    norm, scale = (torch.rand(*shape, generator=g, device="cuda").half() for shape in ((k,), (n, 1)))
    packed = torch.randint(0, 256, (n, k // 2), generator=g, device="cuda").to(torch.uint8)
    ids, logits = torch.zeros(m, dtype=torch.int32, device="cuda"), torch.full((m, n), float("nan"), device="cuda").half()
    torch.cuda.synchronize()
    wrap = lambda t: runtime.wrap(t.data_ptr(), t.numel() * t.element_size())
    runtime.dispatch("llmopt_w4a16_lm_head_argmax_extra_f16", [wrap(t) for t in (x, norm, packed, scale, ids, logits)],
                     u32s(m, n, k) + struct.pack("<f", 1e-5), (256, 1, 1), (256, 1, 1))
    q = torch.stack([packed & 15, packed >> 4], dim=-1).reshape(n, k).double()
    weight = torch.where(q >= 8, q - 16, q) * scale.double()
    rows = x.double() / torch.sqrt(x.double().square().mean(1, keepdim=True) + 1e-5) * norm.double()
    expected = rows @ weight.T
    sums = 2 * 64 * 2.0 ** -24 * 1040 * rows.abs().sum(1, keepdim=True) * scale.double().T
    assert ((logits.double() - expected).abs() <= 2.0 ** -11 * expected.abs() + sums).all()
    chosen = expected.gather(1, ids.long()[:, None])[:, 0]
    assert (chosen >= expected.max(1).values - 2 * sums.max(1).values).all()
    runtime.close()


# One launch that normalises its rows: one to twelve scale groups, an odd and an even number of them, remainders of rows and
# columns, a row of zeros and one of the largest values
NORMED_PAIRS = [(300, 200, 64), (130, 1500, 192), (300, 401, 448), (100, 1537, 576), (129, 1000, 640), (140, 801, 768)]


@pytest.mark.parametrize("m,n,k", NORMED_PAIRS)
def test_pairs_of_rows_that_are_normalised_in_the_tile(runtime, m, n, k):
    """Bit for bit what the norm and the pair leave as launches of their own."""
    rng = np.random.default_rng(m + n + k)
    x, gate, gate_scale, _ = w4_case(rng, m, n, k)
    _, up, up_scale, _ = w4_case(rng, 1, n, k)
    x[m // 2], x[m - 1] = 0, 65504
    norm = rng.uniform(0.5, 1.5, k).astype(np.float16)
    put = runtime.buffer_of_bytes
    params, weights = u32s(m, n, k) + struct.pack("<f", 1e-5), [put(a) for a in (gate, gate_scale, up, up_scale)]
    normed, (one, two) = put(np.zeros((m, k), dtype=np.float16)), (put(np.full((m, n), np.nan, dtype=np.float16)) for _ in range(2))
    runtime.dispatch("llmopt_w4a16_swiglu_rms_f16_g64", [put(x), put(norm), normed], params, (m, 1, 1), (256, 1, 1))
    grid = (linear_grid(((m + 3) // 4) * n), 1, 1)
    runtime.dispatch("llmopt_w4a16_dual_swiglu_f16_g64_m4", [normed, *weights, two], params, grid, (256, 1, 1))
    runtime.dispatch("llmopt_rms_w4a16_dual_swiglu_f16_g64", [put(x), put(norm), *weights, one], params, grid, (256, 1, 1))
    np.testing.assert_array_equal(one.numpy(np.uint16), two.numpy(np.uint16))
    assert np.isfinite(one.numpy(np.float16)).all()


# 256 x 256 tiles (test_tile_rules.py checks which sizes take them): one to nine K steps, remainders of rows and columns, whole and odd rows of outputs and addends
@pytest.mark.parametrize("m,n,k,addend", [(4000, 4100, 64, "none"), (4001, 4097, 128, "bias"), (2050, 7301, 192, "residual"),
                                          (2300, 7304, 256, "residual"), (4096, 4096, 320, "bias"), (2049, 7425, 576, "none"),
                                          (1290, 5889, 192, "bias")])
def test_tiles_of_256(runtime, m, n, k, addend):
    test_small_tiles(runtime, m, n, k, addend)


@pytest.mark.parametrize("m,n,k,addend", [(1290, 5637, 192, "bias")])
def test_tiles_of_128_by_256(runtime, m, n, k, addend):
    test_small_tiles(runtime, m, n, k, addend)


def test_tiles_of_256_keep_infinities_in_their_row(runtime):
    m, n, k = 4001, 4099, 192
    rng = np.random.default_rng(1)
    x, packed, _, _ = w4_case(rng, m, n, k)
    x = rng.integers(-4, 5, (m, k)).astype(np.float16)
    scale = np.ones((n, k // 64), dtype=np.float16)
    expected = product(x, packed, scale)
    np.testing.assert_array_equal(run_linear(runtime, x, packed, scale), expected.astype(np.float16))
    x[m - 1, k - 1] = np.inf
    out = run_linear(runtime, x, packed, scale)
    assert not np.isfinite(out[m - 1]).any()
    np.testing.assert_array_equal(out[:m - 1], expected.astype(np.float16)[:m - 1])


@pytest.mark.parametrize("m,n,k", [(4000, 2100, 64), (4001, 2049, 128), (2050, 3701, 192), (2300, 3704, 320), (2049, 3713, 576)])
def test_pair_tiles_of_256(runtime, m, n, k):
    test_small_pair_tiles(runtime, m, n, k)
