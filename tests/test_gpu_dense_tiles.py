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
# 128 x 192, 256 x 256
@pytest.mark.parametrize("m,n,k", [(2, 5, 64), (33, 700, 192), (500, 2000, 64), (700, 1023, 128), (1023, 2047, 64),
                                   (2047, 2045, 192), (1500, 6001, 64), (2999, 2046, 128), (2047, 8570, 64),
                                   (2046, 6200, 128), (3000, 9503, 64)])
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
                                        (2047, 64, 4285), (3000, 64, 3999)])
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
