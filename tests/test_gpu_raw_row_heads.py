"""One token's attention over a raw row: the query heads of a key head, of which a wave asks for two ahead of the keys, the rest and
groups beyond sixteen later.  A head's result is that of a call with this head alone, bit for bit, and close to float64's."""
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
    norms = bits(2, dim)
    q_norm, k_norm = put(norms[0]), put(norms[1])
    turns = 1e4 ** (-np.arange(max(1, rotated // 2)) / max(1, rotated // 2))
    frequencies = put(turns)

    def call(position, rows):
        row = np.concatenate([rows.reshape(-1), own])
        ring = put(keys), put(values)
        out = put(np.full(len(rows) * vdim, np.nan, dtype=np.float32))
        runtime.dispatch("llmopt_rotary_attention_bf16",
                         [put(row), q_norm, k_norm, frequencies, put(np.array([position, slot], np.uint32)), *ring, out],
                         u32s(1, len(rows), 1, dim, vdim, row.size, len(rows) * vdim, capacity, 0, 1, slots, rotated) +
                         struct.pack("<ffff", dim ** -0.5, 0.0, 1e-6, 1.0), *GRID)
        return out.numpy(np.float32, (len(rows), vdim)), ring[0].numpy(np.uint16), ring[1].numpy(np.uint16)

    exact = lambda b: (b.astype(np.uint32) << 16).view(np.float32).astype(np.float64)

    def turned(vectors, norm, position):
        v = vectors / np.sqrt(np.mean(vectors.astype(np.float64) ** 2, axis=-1, keepdims=True) + 1e-6) * exact(norm)
        half, angle = rotated // 2, position * turns[:rotated // 2]
        low, high = v[..., :half].copy(), v[..., half:rotated].copy()
        v[..., :half], v[..., half:rotated] = low * np.cos(angle) - high * np.sin(angle), high * np.cos(angle) + low * np.sin(angle)
        return v

    for position in (0, 100, 299):
        together = call(position, queries)
        assert np.isfinite(together[0]).all()
        own_key = turned(own[:dim], norms[1], position)
        stored = exact(together[1].reshape(keys.shape)[slot, 0, position])
        assert (np.abs(stored - own_key) <= 2.0 ** -8 * np.abs(own_key) + 1e-6).all()
        q = exact(to_bfloat16(turned(queries, norms[0], position).astype(np.float32)))
        k = np.vstack([exact(keys[slot, 0, :position]), stored[None]])
        v = np.vstack([exact(values[slot, 0, :position]), exact(to_bfloat16(own[dim:]))[None]])
        scores = q @ k.T * dim ** -0.5
        weights = np.exp(scores - scores.max(axis=1, keepdims=True))
        want = weights / weights.sum(axis=1, keepdims=True) @ v
        # The sums' 2^-12 of the largest value (as where the shares are joined); and a query's values within float32's rounding of
        # the middle between two bfloat16 ones may fall the other way, two of a head: a step of 2^-8 each in a score.
        score_off = 2 * 2.0 ** -8 * np.abs(q).max() * np.abs(k).max() * dim ** -0.5
        assert (np.abs(together[0] - want) <= (2.0 ** -12 + np.expm1(2 * score_off)) * np.abs(v).max()).all()
        for head in range(heads):
            alone = call(position, queries[head:head + 1])
            np.testing.assert_array_equal(together[0][head:head + 1], alone[0])
            np.testing.assert_array_equal(together[1], alone[1])
            np.testing.assert_array_equal(together[2], alone[2])
