"""One token's attention where the last workgroup of a key / value head joins its shares of 128 keys, and where a launch of its
own merges them: both sides of the line between them, one live share and the most, several tokens in a row over one set of
arrival counters."""
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


def exact(bits):
    return (bits.astype(np.uint32) << 16).view(np.float32).astype(np.float64)


# 256 and 512 outputs a key head, one more head; value heads of the narrowest form with many queries; rings of 1 to 66 shares
@pytest.mark.parametrize("heads,kv_heads,dim,vdim", [(4, 1, 64, 64), (8, 2, 128, 128), (5, 1, 128, 128), (10, 2, 64, 52), (30, 1, 32, 17),
                                                      (64, 2, 32, 16)])
@pytest.mark.parametrize("capacity", [128, 129, 1024, 1025, 2048, 2049, 8192, 8448])
def test_shares_of_a_token(runtime, heads, kv_heads, dim, vdim, capacity):
    rng = np.random.default_rng(capacity + heads)
    per, slots, slot, scale = heads // kv_heads, 2, 1, np.float32(dim ** -0.5)
    draw = lambda *shape: to_bfloat16(rng.standard_normal(shape, dtype=np.float32))
    q, sink = draw(heads * dim + kv_heads * (dim + vdim)), draw(heads)
    keys, values = draw(slots, kv_heads, capacity, dim), draw(slots, kv_heads, capacity, vdim)
    put = runtime.buffer_of_bytes
    device = [put(a) for a in (q, sink, keys, values)]
    queries = exact(q[:heads * dim]).reshape(kv_heads, per, dim)
    positions = sorted({p for p in (0, 127, 128, 1023, 1024, 2047, 2048, capacity - 1) if p < capacity})
    for has_sink in (0, 1):
        for position in positions + [capacity - 1]:  # (the last once more: the counters were left at zero)
            out = runtime.create_buffer(heads * vdim * 2)
            batch = runtime.begin_batch()
            batch.dispatch("llmopt_chunk_attention_bf16",
                           [device[0], device[1], put(np.array([position, slot], np.uint32)), device[2], device[3], out],
                           u32s(1, heads, kv_heads, dim, vdim, capacity, 0, slots, has_sink) + struct.pack("<ff", scale, 0.0), *GRID)
            batch.commit()
            k, v = exact(keys[slot][:, :position + 1]), exact(values[slot][:, :position + 1])
            scores = np.matmul(queries, k.transpose(0, 2, 1)) * float(scale)
            extra = exact(sink).reshape(kv_heads, per, 1)
            top = np.maximum(scores.max(-1, keepdims=True), extra if has_sink else -np.inf)
            weights = np.exp(scores - top)
            total = weights.sum(-1, keepdims=True) + (np.exp(extra - top) if has_sink else 0.0)
            expected = (np.matmul(weights, v) / total).reshape(-1)
            # the output's rounding to bfloat16 (half a step of 2^-8); weights as two bfloat16 planes (2^-16) of scores that are
            # float32 sums of at most 128 products (2^-14 with room), against the largest value
            bound = 2.0 ** -8 * np.abs(expected) + 2.0 ** -12 * np.abs(v).max()
            got = exact(out.numpy(np.uint16))
            assert (np.abs(got - expected) <= bound).all(), (has_sink, position, np.abs(got - expected).max())
