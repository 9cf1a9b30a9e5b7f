"""A prompt of the gated delta rule in one portion against the same in portions of whole chunks: enough chunks and heads
for three workgroups a compute unit against few enough for two, and every width of the outputs' tiles.  Chunk borders are
the same, so the two differ by the order in which the decays' low-rank products are summed (a few times 2^-24) and the
rounding of an output to bfloat16 that this can move: one unit, 2^-8 of the value."""
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


@pytest.mark.parametrize("m,heads,kv_heads,dim,vdim", [
    (2115, 16, 4, 128, 128), (2070, 16, 16, 72, 40), (2049, 20, 5, 128, 200), (200, 4, 2, 256, 120), (130, 2, 1, 64, 72)])
@pytest.mark.parametrize("kind", ["bf16", "f32"])
def test_one_portion_is_several(runtime, m, heads, kv_heads, dim, vdim, kind):
    rng = np.random.default_rng(m + dim)
    put = runtime.buffer_of_bytes
    taps, ranks, n_out = 4, (8, 16), heads * vdim
    channels = 2 * kv_heads * dim + n_out
    decay_at = (channels + 7) // 8 * 8
    gate_at, ld = decay_at + ranks[0], decay_at + ranks[0] + ranks[1]
    store = to_bfloat16 if kind == "bf16" else (lambda a: a)
    rows = store(rng.standard_normal((m, ld), dtype=np.float32))
    beta = rng.standard_normal((m, heads), dtype=np.float32)
    bf16 = lambda *shape, gain=1.0: put(to_bfloat16(rng.standard_normal(shape, dtype=np.float32) * np.float32(gain)))
    weights = [bf16(heads * dim, ranks[0], gain=ranks[0] ** -0.5), bf16(heads * dim), bf16(heads, gain=0.5),
               bf16(n_out, ranks[1], gain=ranks[1] ** -0.5), bf16(vdim), bf16(channels, taps)]
    results = []
    for portions in ([m], [640] * (m // 640) + [m % 640] if m > 640 else [64, m - 64]):
        ring, state = runtime.create_buffer(taps * channels * 4), put(np.zeros((heads, dim, vdim), dtype=np.float32))
        out, at = [], 0
        for count in portions:
            target = put(np.zeros((count, n_out), dtype=rows.dtype))
            runtime.dispatch(f"llmopt_gated_delta_{kind}",
                             [put(rows[at:at + count]), put(beta[at:at + count]), *weights, ring, state,
                              put(np.array([at, 0], dtype=np.uint32)), target],
                             u32s(count, heads, kv_heads, dim, vdim, taps, 1, ld, 0, decay_at, gate_at, ld, *ranks, n_out, 0) +
                             struct.pack("<ff", 1e-6, 0.5), *GRID)
            part = target.numpy(rows.dtype)
            out.append((from_bfloat16(part) if kind == "bf16" else part).reshape(count, n_out))
            at += count
        results.append((np.concatenate(out), state.numpy(np.float32)))
    (whole, whole_state), (parts, parts_state) = results
    assert np.isfinite(whole).all() and np.abs(whole).max() > 0
    unit = 2.0 ** -8 if kind == "bf16" else 2.0 ** -14
    assert (np.abs(whole - parts) <= unit * np.abs(whole) + 2.0 ** -14 * np.abs(whole).max()).all()
    assert np.abs(whole_state - parts_state).max() <= 2.0 ** -14 * np.abs(whole_state).max()
