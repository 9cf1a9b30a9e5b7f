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


# taps whose inputs are asked for beside the weights (up to four) or not; rows that pass through registers (whole pieces of eight, up
# to 4096) or not; one and two rows a wave
@pytest.mark.parametrize("taps", [1, 2, 4, 5])
@pytest.mark.parametrize("position", [0, 1, 2, 11])
@pytest.mark.parametrize("width,heads,vdim", [(8, 3, 5), (1024, 2, 8), (4096, 3, 5), (4104, 3, 5), (62, 3, 5), (16, 8, 128)])
def test_projection_and_convolution(runtime, taps, position, width, heads, vdim):
    rng = np.random.default_rng(width * 8 + taps)
    groups, state_size, slots, slot, epsilon = 1, 6, 2, 1, np.float32(1e-5)
    inner = heads * vdim
    channels = inner + 2 * groups * state_size
    n = inner + channels + heads
    stream = rng.standard_normal(width).astype(np.float32)
    (norm_bits, norm), (weight_bits, weights) = bf16(rng, width), bf16(rng, n, width)
    (conv_bits, conv), (bias_bits, bias), (dt_bits, dt_bias) = bf16(rng, channels, taps), bf16(rng, channels), bf16(rng, heads)
    ring = rng.standard_normal((slots, taps, channels)).astype(np.float32)
    put = runtime.buffer_of_bytes
    held, out, unused = put(ring), runtime.create_buffer(n * 4), runtime.create_buffer(heads * 4)
    batch = runtime.begin_batch()
    batch.dispatch("llmopt_rms_ssm_input_bf16",
                   [put(stream), put(norm_bits), put(weight_bits), put(np.array([position, slot] + [0] * 6, np.uint32)), put(conv_bits),
                    put(bias_bits), put(dt_bits), held, out, unused],
                   u32s(1, width, heads, vdim, groups, state_size, taps, slots) + epsilon.tobytes(), *GRID)
    batch.commit()
    x = stream.astype(np.float64)
    normed = x / np.sqrt(np.mean(x * x) + float(epsilon)) * norm
    projected = weights @ normed
    # the product's sum of `width` terms, and a few roundings of each term
    error = (width + 16) * ULP * (np.abs(weights) @ np.abs(normed))
    v, dv = projected[inner:inner + channels], error[inner:inner + channels]
    total, size, dtotal = bias + conv[:, -1] * v, np.abs(bias) + np.abs(conv[:, -1] * v), np.abs(conv[:, -1]) * dv
    for back in range(1, min(taps - 1, position) + 1):
        past = conv[:, taps - 1 - back] * ring[slot, (position - back) % taps]
        total, size = total + past, size + np.abs(past)
    dtotal = dtotal + (taps + 2) * ULP * size
    expected, bound = projected.copy(), error.copy()
    expected[inner:inner + channels] = total / (1.0 + np.exp(-total))
    bound[inner:inner + channels] = 1.1 * dtotal + 8 * ULP * np.abs(total) * (1.0 + np.abs(total))  # (silu's slope is at most 1.1)
    z = projected[inner + channels:] + dt_bias
    expected[inner + channels:] = np.log1p(np.exp(-np.abs(z))) + np.maximum(z, 0.0)
    bound[inner + channels:] += 8 * ULP * (1.0 + np.abs(z))
    assert (np.abs(out.numpy(np.float32) - expected) <= bound).all()
    kept = held.numpy(np.float32, ring.shape)
    assert (np.abs(kept[slot, position % taps] - v) <= dv).all()
    ring[slot, position % taps] = kept[slot, position % taps]
    assert (kept == ring).all()
