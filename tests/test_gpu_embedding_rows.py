"""Rows of the bfloat16 embedding table as scaled float32: whole pieces of eight values or not, one workgroup a row and more, tokens
outside the table."""
import struct

import numpy as np
import pytest

from llmopt_amd.safetensors_file import to_bfloat16
from tests.gpu_util import u32s

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def runtime():
    from llmopt_amd.native import Runtime
    rt = Runtime()
    yield rt
    rt.close()


@pytest.mark.parametrize("width", [1, 7, 8, 16, 2040, 2048, 2056, 2049, 4104])
@pytest.mark.parametrize("tokens", [[5], [0, 36, 37, -1, 12, 1 << 40]])
def test_rows_of_the_table(runtime, width, tokens):
    rng = np.random.default_rng(width)
    vocabulary, scale = 37, np.float32(1.7)
    table = to_bfloat16(rng.standard_normal((vocabulary, width), dtype=np.float32))
    out = runtime.buffer_of_bytes(np.full((len(tokens), width), np.nan, np.float32))
    runtime.dispatch("llmopt_embedding_scaled_bf16",
                     [runtime.buffer_of_bytes(np.array(tokens, np.int64)), runtime.buffer_of_bytes(table), out],
                     u32s(len(tokens), vocabulary, width) + struct.pack("<f", scale), (1, 1, 1), (256, 1, 1))
    rows = (table.astype(np.uint32) << 16).view(np.float32) * scale
    expected = np.stack([rows[t] if 0 <= t < vocabulary else np.zeros(width, np.float32) for t in tokens])
    np.testing.assert_array_equal(out.numpy(np.float32, expected.shape), expected)
