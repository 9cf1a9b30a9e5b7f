"""One token through window attention and the gated delta rule as one entry against the two entries one after the other:
the attention's rows and rings bit for bit, the delta rule's row and state up to the float32 rounding of sums taken in
another order (a few units in the last place of values of order one, over up to 256 terms)."""
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


# heads, kv_heads, dim, vdim, window, rotated | heads, kv_heads, dim, vdim | ranks | positions
@pytest.mark.parametrize("left,right,ranks,positions", [
    ((16, 4, 64, 64, 2048, 64), (8, 8, 128, 128), (128, 128), (0, 1, 127, 128, 700)),
    ((16, 4, 128, 128, 512, 128), (16, 16, 128, 128), (128, 64), (0, 300, 511, 512, 4000)),
    ((6, 2, 40, 48, 96, 14), (4, 2, 100, 32), (8, 24), (0, 95, 96, 97)),
    ((9, 3, 64, 128, 0, 0), (3, 1, 256, 96), (16, 128), (0, 5, 900)),
    ((4, 1, 128, 64, 130, 64), (2, 2, 20, 256), (72, 8), (3, 129, 130)),
    ((4, 2, 256, 64, 200, 64), (2, 2, 64, 64), (128, 128), (0, 250)),   # attention heads too wide for the shared launch
    ((4, 2, 64, 64, 200, 64), (2, 2, 64, 40), (128, 128), (0, 250)),    # value columns in no whole parts
    ((4, 2, 64, 64, 200, 64), (2, 2, 64, 64), (12, 136), (0, 250)),     # ranks in no whole pieces, and too long
])
def test_one_entry_is_the_two(runtime, left, right, ranks, positions):
    rng = np.random.default_rng(hash((left, right)) % (1 << 32))
    heads, kv, dim, vdim, window, rotated = left
    d_heads, d_kv, d_dim, d_vdim = right
    taps, slots, slot, capacity = 4, 3, 2, window or 1024
    up = lambda n: (n + 7) // 8 * 8
    channels = 2 * d_kv * d_dim + d_heads * d_vdim
    conv = up(heads * dim + kv * (dim + vdim))
    decay_at = up(conv + channels)
    gate_at = up(decay_at + ranks[0])
    split = up(gate_at + ranks[1])
    n_left, n_right = heads * vdim, d_heads * d_vdim
    put = runtime.buffer_of_bytes
    bf16 = lambda *shape, gain=1.0: put(to_bfloat16(rng.standard_normal(shape, dtype=np.float32) * np.float32(gain)))
    row = rng.standard_normal(split + d_heads).astype(np.float32)
    q_norm, k_norm, norm = bf16(dim), bf16(dim), bf16(d_vdim)
    frequencies = put(1e4 ** (-np.arange(max(1, rotated // 2)) / max(1, rotated // 2)))
    w_decay, w_gate = (bf16(size, rank, gain=rank ** -0.5) for size, rank in ((d_heads * d_dim, ranks[0]), (n_right, ranks[1])))
    dt_bias, a_log, conv_w = bf16(d_heads * d_dim), bf16(d_heads, gain=0.5), bf16(channels, taps)
    keys = to_bfloat16(rng.standard_normal((slots, kv, capacity, dim), dtype=np.float32))
    values = to_bfloat16(rng.standard_normal((slots, kv, capacity, vdim), dtype=np.float32))
    state = rng.standard_normal((slots, d_heads, d_dim, d_vdim)).astype(np.float32)
    conv_ring = runtime.create_buffer(slots * taps * channels * 4)
    eps = struct.pack("<f", 1e-6)
    attention_parameters = u32s(1, heads, kv, dim, vdim, split, n_left + n_right, capacity, window, 1, slots, rotated) + \
        struct.pack("<ff", dim ** -0.5, 0.0) + eps + struct.pack("<f", 0.7)
    delta_parameters = u32s(1, d_heads, d_kv, d_dim, d_vdim, taps, slots, split, conv, decay_at, gate_at, split, *ranks,
                            n_left + n_right, n_left) + eps + struct.pack("<f", 0.3)
    for position in positions:
        left_over = []
        for together in (False, True):
            b_row, b_out = put(row), put(np.full(n_left + n_right, np.nan, dtype=np.float32))
            b_keys, b_values, b_state, step = put(keys), put(values), put(state), put(np.array([position, slot], dtype=np.uint32))
            attention = [b_row, q_norm, k_norm, frequencies, step, b_keys, b_values, b_out]
            delta = [b_row, b_row, w_decay, dt_bias, a_log, w_gate, norm, conv_w, conv_ring, b_state, step, b_out]
            if together:
                runtime.dispatch("llmopt_rotary_attention_gated_delta_bf16", attention + delta[2:10],
                                 attention_parameters + delta_parameters, *GRID)
            else:
                runtime.dispatch("llmopt_rotary_attention_bf16", attention, attention_parameters, *GRID)
                runtime.dispatch("llmopt_gated_delta_bf16", delta, delta_parameters, *GRID)
            left_over.append([b_out.numpy(np.float32), b_keys.numpy(np.uint16), b_values.numpy(np.uint16),
                              b_state.numpy(np.float32)])
        two, one = left_over
        np.testing.assert_array_equal(one[0][:n_left], two[0][:n_left])
        np.testing.assert_array_equal(one[1], two[1])
        np.testing.assert_array_equal(one[2], two[2])
        for got, expected in ((one[0][n_left:], two[0][n_left:]), (one[3], two[3])):
            assert np.isfinite(got).all()
            assert np.abs(got - expected).max() <= 256 * 2.0 ** -24 * max(1.0, np.abs(expected).max()), position
