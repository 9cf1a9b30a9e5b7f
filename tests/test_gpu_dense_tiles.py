"""The tiles of the bfloat16 product, each at sizes with remainders of rows and columns, against float64."""
import struct

import numpy as np
import pytest

from llmopt_amd.safetensors_file import from_bfloat16, to_bfloat16
from tests.gpu_util import u32s

pytestmark = pytest.mark.gpu
GRID = ((1, 1, 1), (256, 1, 1))


@pytest.fixture(scope="module")
def runtime():
    from llmopt_amd.native import Runtime
    rt = Runtime()
    yield rt
    rt.close()


def values(rng, *shape, gain=1.0):
    patterns = to_bfloat16(rng.standard_normal(shape, dtype=np.float32) * np.float32(gain))
    return patterns, from_bfloat16(patterns).reshape(shape).astype(np.float64)


# 32 x 64, 64 x 64, 64 x 128, 128 x 128 with eight and with four waves, 192 x 128 with eight and with four,
# 128 x 192, 256 x 256, 64 x 128 with four waves (test_tile_rules.py checks which sizes take which)
@pytest.mark.parametrize("m,n,k", [(2, 5, 64), (33, 700, 192), (500, 2000, 64), (700, 1023, 128), (1023, 2047, 64),
                                   (2047, 2045, 192), (1500, 6001, 64), (2999, 2046, 128), (2047, 8570, 64),
                                   (2046, 6200, 128), (3000, 9503, 64), (1000, 5551, 64), (1000, 6357, 64), (2047, 2045, 64),
                                   (1499, 2047, 256), (1345, 8857, 256), (1413, 8123, 256), (195, 8311, 2560),
                                   (203, 8125, 2304)])
def test_tiles(runtime, m, n, k):
    rng = np.random.default_rng(m + n + k)
    (x, fx), (w, fw) = values(rng, m, k), values(rng, n, k)
    out = runtime.buffer_of_bytes(np.full((m, n), np.nan, dtype=np.float32))
    runtime.dispatch("llmopt_linear_store_bf16", [runtime.buffer_of_bytes(x), runtime.buffer_of_bytes(w), out], u32s(m, n, k),
                     *GRID)
    error = np.abs(out.numpy(np.float32, (m, n)) - fx @ fw.T)
    # exact products, k float32 additions, each within a unit in the last place of a sum of magnitudes
    assert np.all(error <= 2.0 * k * 2.0 ** -24 * (np.abs(fx) @ np.abs(fw).T))


@pytest.mark.parametrize("m,width,ff", [(40, 128, 300), (500, 128, 1000), (700, 64, 3000), (1023, 128, 1500),
                                        (2047, 64, 4285), (3000, 64, 3999), (500, 64, 1210), (1000, 64, 2827),
                                        (1000, 64, 3230), (2047, 64, 3129), (1023, 64, 1500), (1345, 256, 4429),
                                        (1413, 256, 4061), (195, 2560, 4155), (203, 2304, 4062)])
def test_gated_tiles(runtime, m, width, ff):
    """Norm, gated pair and down projection: what is rounded to bfloat16 between them (the normed rows and the products,
    half a unit, 2^-9, each) shows in the output at that size."""
    rng = np.random.default_rng(m + ff)
    stream = rng.standard_normal((m, width)).astype(np.float32)
    norm, fnorm = values(rng, width)
    (gate, fgate), (up, fup) = values(rng, ff, width, gain=width ** -0.5), values(rng, ff, width, gain=width ** -0.5)
    down, fdown = values(rng, width, ff, gain=ff ** -0.5)
    out = runtime.buffer_of_bytes(stream)
    runtime.dispatch("llmopt_rms_gated_ffn_add_bf16", [out] + [runtime.buffer_of_bytes(a) for a in (norm, gate, up, down)],
                     u32s(m, width, ff) + struct.pack("<f", 1e-6) + u32s(0), *GRID)
    x = stream.astype(np.float64)
    h = x / np.sqrt(np.mean(x * x, axis=1, keepdims=True) + 1e-6) * fnorm
    g = h @ fgate.T
    expected = (g / (1.0 + np.exp(-g)) * (h @ fup.T)) @ fdown.T
    error = out.numpy(np.float32, (m, width)) - x - expected
    assert np.sqrt(np.mean(error ** 2)) <= 4 * 2.0 ** -9 * np.sqrt(np.mean(expected ** 2))


def test_gate_whose_reciprocal_is_no_normal_number(runtime):
    """silu(-88) = -88 / (1 + e^88) = -5.3e-37, whose quotient is one and whose reciprocal, 6e-39, is less than the smallest normal
    float32.  An up half of 1e36 shows it; bfloat16 rounds gate, up, product and row, half a unit (2^-9) each, and e^88 is good to
    88 log2(e) 2^-24 ln(2) < 2^-17."""
    m, width = 40, 64
    column = np.zeros((width, width), dtype=np.float32)
    column[:, 0] = 1.0
    put, bf16 = runtime.buffer_of_bytes, lambda v: to_bfloat16(v.astype(np.float32))
    norm, gate, up, down = bf16(np.ones(width)), bf16(-88.0 * column), bf16(1e36 * column), bf16(np.eye(width))
    out = put(np.ones((m, width), dtype=np.float32))
    runtime.dispatch("llmopt_rms_gated_ffn_add_bf16", [out] + [put(a) for a in (norm, gate, up, down)],
                     u32s(m, width, width) + struct.pack("<f", 1e-9) + u32s(0), *GRID)
    expected = -88.0 / (1.0 + np.exp(88.0)) * float(from_bfloat16(bf16(np.array([1e36])))[0])
    got = out.numpy(np.float32, (m, width)).astype(np.float64) - 1.0
    assert np.all(np.abs(got - expected) <= 4 * 2.0 ** -9 * abs(expected))


ROW_SIZES = [(33, 701, 64), (500, 2000, 64), (1023, 2047, 64), (2047, 2045, 64), (1000, 5551, 64), (1000, 6357, 64),
             (1500, 6001, 64), (2999, 2046, 64), (3000, 9503, 64), (1499, 2047, 256), (1345, 8857, 256), (1413, 8123, 256),
             (195, 8311, 2560), (203, 8125, 2304)]


def normed(rng, m, k):
    stream = rng.standard_normal((m, k)).astype(np.float32)
    norm, fnorm = values(rng, k)
    x = stream.astype(np.float64)
    return stream, norm, x / np.sqrt(np.mean(x * x, axis=1, keepdims=True) + 1e-6) * fnorm


def assert_rows(got, h, weight, mixed=None):
    """A normed value is rounded to bfloat16 before the product and the result after it: seven fraction bits, half a unit is
    up to 2^-8 of the value; 2^-12 for the norm's and the sums' float32."""
    expected = h @ weight.T
    bound = (2.0 ** -8 + 2.0 ** -12) * (np.abs(h) @ np.abs(weight).T)
    if mixed is not None:
        expected = (expected + mixed) / 2  # (a half of each)
    assert got.shape == expected.shape and np.isfinite(got).all()
    assert np.all(np.abs(got - expected) <= bound + (2.0 ** -8 + 2.0 ** -12) * np.abs(expected))


@pytest.mark.parametrize("m,n,k", ROW_SIZES)
def test_rows_with_mixed_values(runtime, m, n, k):
    """bfloat16 rows out of every tile: QKV, whose last columns are mixed with another layer's."""
    rng = np.random.default_rng(m + n)
    stream, norm, h = normed(rng, m, k)
    weight, fweight = values(rng, n, k, gain=k ** -0.5)
    first = rng.standard_normal((m, n - 16)).astype(np.float32)
    put = runtime.buffer_of_bytes
    out = put(np.full((m, n), 0x7fc0, dtype=np.uint16))  # NaN
    rings = [put(np.zeros(size, dtype=np.uint16)) for size in (8, n - 16)]
    runtime.dispatch("llmopt_rms_qkv_chunk_bf16", [put(stream), put(norm), put(weight), put(np.zeros(2, dtype=np.uint32)), out,
                                                   put(first), *rings],
                     u32s(m, k, 1, 1, 8, n - 16) + struct.pack("<fIf", 1e-6, 2, 0.5) + u32s(1, 1, 1), *GRID)
    got = from_bfloat16(out.numpy(np.uint16)).reshape(m, n).astype(np.float64)
    assert_rows(got[:, :16], h, fweight[:16])
    assert_rows(got[:, 16:], h, fweight[16:], first.astype(np.float64))


@pytest.mark.parametrize("m,n,k", ROW_SIZES)
def test_rows_split_in_two(runtime, m, n, k):
    """The same with the last columns, a time step a head, as float32 in an array of their own."""
    rng = np.random.default_rng(m * 3 + n)
    heads, vdim = (5, 3) if n % 2 else (4, 3)
    states = (n - heads - 2 * heads * vdim) // 2
    columns, channels = n - heads, heads * vdim + 2 * states
    stream, norm, h = normed(rng, m, k)
    weight, fweight = values(rng, n, k, gain=k ** -0.5)
    put = runtime.buffer_of_bytes
    zeros = lambda size, dtype: put(np.zeros(size, dtype=dtype))
    out, steps = put(np.full((m, columns), 0x7fc0, dtype=np.uint16)), put(np.full((m, heads), np.nan, dtype=np.float32))
    runtime.dispatch("llmopt_rms_ssm_input_bf16",
                     [put(stream), put(norm), put(weight), zeros(2, np.uint32), zeros(channels * 4, np.uint16),
                      zeros(channels, np.uint16), zeros(heads, np.uint16), zeros(channels * 4, np.float32), out, steps],
                     u32s(m, k, heads, vdim, 1, states, 4, 1) + struct.pack("<f", 1e-6), *GRID)
    assert_rows(from_bfloat16(out.numpy(np.uint16)).reshape(m, columns).astype(np.float64), h, fweight[:columns])
    assert_rows(steps.numpy(np.float32, (m, heads)).astype(np.float64), h, fweight[columns:])


# Tiles whose waves multiply and read at different times: 256 x 256, in turns 192 x 128, 128 x 128, 128 x 192, 256 x 128 and
# 128 x 64, each with remainders, an even and an odd number of stages (test_tile_rules.py checks which sizes take which)
STAGGERED = [(1030, 10967, 1024), (1345, 8853, 1088), (3000, 1500, 1280), (1345, 3001, 1344), (1345, 1500, 1792),
             (200, 9503, 1856), (500, 9503, 1280), (500, 9503, 1344), (1345, 5001, 1280), (1345, 5001, 1344),
             (257, 4095, 1280), (200, 5001, 1344)]
# two launches: whole rounds of 256 x 256, then 64 x 64 or smaller ones, and in turns
SPLIT = [(2047, 8300, 1024), (2047, 9503, 1344), (2047, 9503, 1792)]
# columns that are no whole pieces, where whole ones take 256 x 256
ODD = [(1345, 6001, 1024), (3000, 3001, 1088)]
# 128 x 128 tiles in step up to K = 1791
SHORT = [(1345, 1500, 1280), (200, 9503, 1344)]


@pytest.mark.parametrize("m,n,k", STAGGERED + SPLIT + ODD + SHORT)
def test_staggered_tiles(runtime, m, n, k):
    test_tiles(runtime, m, n, k)


@pytest.mark.parametrize("m,n,k", STAGGERED + SPLIT + ODD + SHORT)
def test_staggered_tiles_of_rows(runtime, m, n, k):
    test_rows_with_mixed_values(runtime, m, n, k)


@pytest.mark.parametrize("m,n,k", STAGGERED + SPLIT + ODD + SHORT)
def test_staggered_tiles_of_pairs(runtime, m, n, k):
    test_gated_tiles(runtime, m, k, n // 2)


# tiles of 128 rows of an expert, in turns and (more than a round of them) in step: 1 to 5 stages and 16, experts with a remainder
@pytest.mark.parametrize("m,width,ff", [(200, 64, 128), (400, 128, 64), (333, 192, 320), (250, 256, 192), (1024, 1024, 320),
                                        (1500, 512, 1600), (1024, 2048, 64)])
def test_routed_tiles(runtime, m, width, ff):
    rng = np.random.default_rng(m + ff)
    experts, top = 5, 2
    stream = rng.standard_normal((m, width)).astype(np.float32)
    norm, fnorm = values(rng, width)
    router, frouter = values(rng, experts, width, gain=width ** -0.5)
    (gate, fgate), (up, fup) = (values(rng, experts, ff, width, gain=width ** -0.5) for _ in range(2))
    down, fdown = values(rng, experts, width, ff, gain=ff ** -0.5)
    put = runtime.buffer_of_bytes
    out, none = put(stream), put(np.zeros(width, dtype=np.uint16))
    runtime.dispatch("llmopt_rms_routed_ffn_add_bf16", [out] + [put(a) for a in (norm, router, gate, up, down)] + [none] * 3,
                     u32s(m, width, experts, top, ff, 0) + struct.pack("<f", 1e-6) + u32s(0), *GRID)
    x = stream.astype(np.float64)
    h = x / np.sqrt(np.mean(x * x, axis=1, keepdims=True) + 1e-6) * fnorm
    scores = h @ frouter.T
    order = np.sort(scores, axis=1)
    clear = order[:, -top] - order[:, -top - 1] > 0.1  # (a close call may go the other way with rounded rows)
    chosen = np.argsort(-scores, axis=1)[:, :top]
    weights = np.exp(np.take_along_axis(scores, chosen, 1))
    weights /= weights.sum(axis=1, keepdims=True)
    expected = np.zeros_like(x)
    for e in range(experts):
        g = h @ fgate[e].T
        y = (g / (1.0 + np.exp(-g)) * (h @ fup[e].T)) @ fdown[e].T
        expected += np.where(chosen == e, weights, 0.0).sum(axis=1, keepdims=True) * y
    error = (out.numpy(np.float32, (m, width)) - x - expected)[clear]
    # normed rows, products and an expert's outputs are rounded to bfloat16 (half a unit, 2^-9, each), and the weights of the
    # experts follow from scores of rounded rows
    assert clear.sum() > m // 2 and np.sqrt(np.mean(error ** 2)) <= 6 * 2.0 ** -9 * np.sqrt(np.mean(expected[clear] ** 2))


def test_split_columns_of_steps(runtime):
    test_rows_split_in_two(runtime, *SPLIT[0])


# The logits of one row among several: short rows, more than 4096 values, no whole pieces of four or eight
@pytest.mark.parametrize("m,width,vocabulary,row", [(5, 64, 100, 3), (2, 2048, 1001, 0), (700, 1000, 333, 699), (3, 4104, 50, 1),
                                                    (4, 1001, 77, 2)])
@pytest.mark.parametrize("pending", [False, True])
def test_logits_of_one_row(runtime, m, width, vocabulary, row, pending):
    """Float32 sums of `width` products: 2^-24 of a sum of magnitudes each, a few units for the norms and the cap."""
    rng = np.random.default_rng(m + width)
    x, y = (rng.standard_normal((m, width)).astype(np.float32) for _ in range(2))
    (add, fadd), (norm, fnorm), (head, fhead) = values(rng, width), values(rng, width), values(rng, vocabulary, width, gain=width ** -0.5)
    put, rms = runtime.buffer_of_bytes, lambda v: v / np.sqrt(np.mean(v * v) + 1e-6)
    out, index = put(np.full(vocabulary, np.nan, dtype=np.float32)), put(np.array([row], dtype=np.uint32))
    stream = x[row].astype(np.float64)
    if pending:
        stream = stream + 0.5 * rms(y[row].astype(np.float64)) * (1.0 + fadd)
        normed = rms(stream) * (1.0 + fnorm)
        runtime.dispatch("llmopt_pending_logits_bf16", [put(x), put(y), put(add), put(x), index, put(norm), put(head), out],
                         u32s(1, width, vocabulary, m, 1) + struct.pack("<4f", 1e-6, 1.0, 0.5, 30.0), *GRID)
    else:
        normed = rms(stream) * fnorm
        runtime.dispatch("llmopt_rms_logits_bf16", [put(x), index, put(norm), put(head), out],
                         u32s(1, width, vocabulary) + struct.pack("<fI", 1e-6, m), *GRID)
    expected = fhead @ normed
    bound = (width + 16) * 2.0 ** -24 * (np.abs(fhead) @ np.abs(normed))
    if pending:
        expected, bound = 30.0 * np.tanh(expected / 30.0), bound + 16 * 2.0 ** -24 * 30.0
    assert np.all(np.abs(out.numpy(np.float32) - expected) <= bound)
