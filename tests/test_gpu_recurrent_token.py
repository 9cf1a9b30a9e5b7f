"""One token through the Mamba-2 recurrence, at the edges of the forms that its kernels take, against float64."""
import numpy as np
import pytest

from llmopt_amd.safetensors_file import to_bfloat16
from tests.gpu_util import u32s

pytestmark = pytest.mark.gpu
GRID = ((1, 1, 1), (256, 1, 1))
ULP = 2.0 ** -24


@pytest.fixture(scope="module")
def runtime():
    from llmopt_amd.native import Runtime
    rt = Runtime()
    yield rt
    rt.close()


def bf16(rng, *shape):
    bits = to_bfloat16(rng.standard_normal(shape, dtype=np.float32))
    return bits, (bits.astype(np.uint32) << 16).view(np.float32).astype(np.float64)


# whole pieces of four values, one and two a lane (up to 128, up to 256) or not; rows that fill their workgroups of eight or not
@pytest.mark.parametrize("state_size", [4, 8, 124, 128, 132, 252, 256, 2, 127, 130, 255])
@pytest.mark.parametrize("heads,vdim,groups", [(1, 1, 1), (3, 4, 3), (4, 6, 2), (6, 3, 1), (8, 64, 2)])
@pytest.mark.parametrize("position", [0, 9])
def test_state_and_output(runtime, state_size, heads, vdim, groups, position):
    rng = np.random.default_rng(state_size * 64 + heads)
    inner, slots, slot = heads * vdim, 3, 1
    channels = inner + 2 * groups * state_size
    row = rng.standard_normal(inner + channels + heads).astype(np.float32)
    row[inner + channels:] = rng.uniform(0.01, 2.0, heads)  # (behind its softplus)
    state = rng.standard_normal((slots, inner, state_size)).astype(np.float32)
    (rate_bits, rate), (skip_bits, skip) = bf16(rng, heads), bf16(rng, heads)
    put = runtime.buffer_of_bytes
    held, out = put(state), runtime.create_buffer(inner * 4)
    unused = put(np.zeros(channels * 4, np.float32))
    batch = runtime.begin_batch()
    batch.dispatch("llmopt_ssm_mix_bf16",
                   [put(np.array([position, slot] + [0] * 6, np.uint32)), put(row), unused, unused, unused, unused, put(rate_bits),
                    put(skip_bits), put(np.zeros(slots * channels, np.float32)), held, out],
                   u32s(1, heads, vdim, groups, state_size, 1, slots), *GRID)
    batch.commit()

    z, x, dt = (row[:inner].astype(np.float64), row[inner:2 * inner].astype(np.float64), row[inner + channels:].astype(np.float64))
    b, c = row[2 * inner:inner + channels].astype(np.float64).reshape(2, groups, state_size)
    head = np.arange(inner) // vdim
    group = head // (heads // groups)
    decayed = np.exp(-np.exp(rate) * dt)[head, None] * state[slot] * (position > 0)
    added = (dt[head] * x)[:, None] * b[group]
    expected = state.astype(np.float64)
    expected[slot] = decayed + added
    # The exponent is off by a few roundings of its size, the sum by a few of its terms'.
    size = np.abs(decayed) * (1.0 + (np.exp(rate) * dt)[head, None]) + np.abs(added)
    kept = held.numpy(np.float32, state.shape)
    assert (np.abs(kept[slot] - expected[slot]) <= 8 * ULP * size).all()
    assert (kept[[0, 2]] == state[[0, 2]]).all()
    gate = z / (1.0 + np.exp(-z))
    y = ((expected[slot] * c[group]).sum(-1) + skip[head] * x) * gate
    # a sum of state_size products and one, and the gate's quotient and exponential
    bound = (state_size + 32) * ULP * ((size * np.abs(c[group])).sum(-1) + np.abs(skip[head] * x)) * np.abs(gate) * (1.0 + np.abs(z))
    assert (np.abs(out.numpy(np.float32) - y) <= bound + 1e-30).all()
