"""One token's attention over a raw row: the query heads of a key head, of which a wave asks for two ahead of the keys, the rest and
groups beyond sixteen later.  A head's result is that of a call with this head alone, bit for bit."""
import struct

import numpy as np
import pytest

from llmopt_amd.safetensors_file import to_bfloat16
from tests.gpu_util import u32s

pytestmark = pytest.mark.gpu
GRID = ((1, 1, 1), (256, 1, 1))


@pytest.fixture(scope="module")
def runtime():
    from llmopt_amd.native import Runtime
    rt = Runtime()
    yield rt
    rt.close()


# up to three vectors with the key, one and two a wave, one more, sixteen, more than sixteen
@pytest.mark.parametrize("heads", [1, 2, 3, 4, 7, 8, 15, 16, 17, 35])
@pytest.mark.parametrize("dim,vdim,rotated", [(64, 64, 64), (128, 128, 64), (40, 48, 14), (64, 48, 0)])
def test_heads_do_not_depend_on_each_other(runtime, heads, dim, vdim, rotated):
    rng = np.random.default_rng(heads * 1000 + dim + vdim)
    slots, slot, capacity = 2, 1, 300
    bits = lambda *shape: to_bfloat16(rng.standard_normal(shape, dtype=np.float32))
    put = runtime.buffer_of_bytes
    queries, own = rng.standard_normal((heads, dim)).astype(np.float32), rng.standard_normal(dim + vdim).astype(np.float32)
    keys, values = bits(slots, 1, capacity, dim), bits(slots, 1, capacity, vdim)
    q_norm, k_norm = put(bits(dim)), put(bits(dim))
    frequencies = put(1e4 ** (-np.arange(max(1, rotated // 2)) / max(1, rotated // 2)))

    def call(position, rows):
        row = np.concatenate([rows.reshape(-1), own])
        ring = put(keys), put(values)
        out = put(np.full(len(rows) * vdim, np.nan, dtype=np.float32))
        runtime.dispatch("llmopt_rotary_attention_bf16",
                         [put(row), q_norm, k_norm, frequencies, put(np.array([position, slot], np.uint32)), *ring, out],
                         u32s(1, len(rows), 1, dim, vdim, row.size, len(rows) * vdim, capacity, 0, 1, slots, rotated) +
                         struct.pack("<ffff", dim ** -0.5, 0.0, 1e-6, 1.0), *GRID)
        return out.numpy(np.float32, (len(rows), vdim)), ring[0].numpy(np.uint16), ring[1].numpy(np.uint16)

    for position in (0, 100, 299):
        together = call(position, queries)
        assert np.isfinite(together[0]).all()
        for head in range(heads):
            alone = call(position, queries[head:head + 1])
            np.testing.assert_array_equal(together[0][head:head + 1], alone[0])
            np.testing.assert_array_equal(together[1], alone[1])
            np.testing.assert_array_equal(together[2], alone[2])
