"""Products over a pending row (a sublayer's output joins the stream behind its norm, the sum is normalised itself) at the edges
of the forms that stage it."""
import struct

import numpy as np
import pytest

from llmopt_amd.safetensors_file import to_bfloat16
from tests.gpu_util import u32s

pytestmark = pytest.mark.gpu
GRID = ((1, 1, 1), (256, 1, 1))
EPSILON, OFFSET, SCALE = np.float32(1e-5), np.float32(1.0), np.float32(0.75)


@pytest.fixture(scope="module")
def runtime():
    from llmopt_amd.native import Runtime
    rt = Runtime()
    yield rt
    rt.close()


def exact(bits):
    return (bits.astype(np.uint32) << 16).view(np.float32).astype(np.float64)


# one piece of four a thread up to 1024, four up to 4096, eight up to 8192; no whole pieces of four, or of eight
@pytest.mark.parametrize("width", [4, 8, 252, 1020, 1024, 1028, 1022, 2048, 4096, 4100, 8192])
@pytest.mark.parametrize("m,row,pending", [(1, 0, True), (5, 3, True), (1, 0, False)])
@pytest.mark.parametrize("suffix", ["_bf16", "_f32"])
def test_logits_of_a_pending_row(runtime, width, m, row, pending, suffix):
    rng = np.random.default_rng(width * 8 + m)
    vocabulary = 37
    stream, output = (rng.standard_normal((m, width)).astype(np.float32) for _ in range(2))
    add, own = (to_bfloat16(rng.standard_normal(width, dtype=np.float32) * np.float32(0.2)) for _ in range(2))
    head = to_bfloat16(rng.standard_normal((vocabulary, width), dtype=np.float32))
    put, out = runtime.buffer_of_bytes, runtime.create_buffer(vocabulary * 4)
    batch = runtime.begin_batch()
    batch.dispatch("llmopt_pending_logits" + suffix,
                   [put(stream), put(output), put(add), runtime.create_buffer(m * width * 4), put(np.array([row], np.uint32)),
                    put(own), put(head), out],
                   u32s(1, width, vocabulary, m, int(pending)) + struct.pack("<ffff", EPSILON, OFFSET, SCALE, 0.0), *GRID)
    batch.commit()
    x = stream[row].astype(np.float64)
    if pending:
        y = output[row].astype(np.float64)
        x = x + y * float(SCALE) / np.sqrt(np.mean(y * y) + float(EPSILON)) * (float(OFFSET) + exact(add))
    normed = x / np.sqrt(np.mean(x * x) + float(EPSILON)) * (float(OFFSET) + exact(own))
    weights = exact(head)
    # float32 sums of `width` products, and a dozen roundings of each value of the row, of the row's size before it cancels
    bound = (width + 16) * 2.0 ** -24 * (np.abs(weights) @ (np.abs(normed) + 2.0))
    assert (np.abs(out.numpy(np.float32) - weights @ normed) <= bound).all()
