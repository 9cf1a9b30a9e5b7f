"""Attention of a portion of a prompt over chunks and windows, at the edges of its tiles: 64 rows whose keys the waves
halve, 128 rows of heads that fill the compute units, four waves for wide heads; against float64 on the same bfloat16
values.  A weighted mean of values is rounded to bfloat16 (2^-9 of itself); its weights carry 17 bits, and scores of
order ten summed in float32 move them by less: 2^-13 of the largest value in all."""
import struct

import numpy as np
import pytest

from llmopt_amd.safetensors_file import from_bfloat16, to_bfloat16
from tests.gpu_util import u32s

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
GRID = ((1, 1, 1), (256, 1, 1))


@pytest.fixture(scope="module")
def runtime():
    from llmopt_amd.native import Runtime
    rt = Runtime()
    yield rt
    rt.close()


# rows, heads, kv_heads, dim, vdim, span, softcap, sink, position of the first row, sliding
@pytest.mark.parametrize("m,heads,kv,dim,vdim,span,softcap,sink,first,sliding", [
    (2, 4, 2, 64, 64, 256, 0.0, True, 0, False),
    (15, 3, 1, 32, 32, 100, 30.0, True, 33, False),
    (16, 4, 4, 64, 32, 64, 50.0, False, 31, False),
    (17, 2, 2, 40, 24, 33, 30.0, True, 32, False),
    (63, 4, 2, 64, 128, 128, 0.0, True, 1, False),
    (64, 4, 2, 128, 128, 4096, 30.0, False, 64, False),
    (65, 4, 2, 128, 64, 96, 0.0, True, 95, False),
    (129, 8, 2, 128, 128, 512, 30.0, True, 127, False),
    (33, 4, 2, 256, 64, 64, 0.0, True, 40, False),
    (70, 2, 1, 64, 256, 64, 30.0, False, 0, False),
    (1025, 32, 8, 128, 128, 700, 30.0, True, 500, False),     # 128-row tiles, bounded scores
    (1153, 32, 4, 72, 48, 2048, 0.0, False, 3, False),        # 128-row tiles of narrower heads
    (1100, 32, 8, 128, 128, 300, 0.0, False, 250, True),      # 128-row tiles, a window
    (300, 6, 2, 64, 64, 97, 0.0, False, 200, True),
    (31, 6, 3, 128, 40, 1, 0.0, False, 5, True),              # a window of one
])
def test_tiles(runtime, m, heads, kv, dim, vdim, span, softcap, sink, first, sliding):
    rng = np.random.default_rng(m * 31 + heads)
    capacity, slots, slot, scale = span, 2, 1, dim ** -0.5
    n = heads * dim + kv * (dim + vdim)
    bf16 = lambda *shape: to_bfloat16(rng.standard_normal(shape, dtype=np.float32))
    rows, sinks = bf16(m, n), bf16(heads)
    ring_k, ring_v = bf16(slots, kv, capacity, dim), bf16(slots, kv, capacity, vdim)
    put = runtime.buffer_of_bytes
    b_rows, b_k, b_v = put(rows), put(ring_k), put(ring_v)
    step, out = put(np.array([first, slot], dtype=np.uint32)), runtime.create_buffer(m * heads * vdim * 2)
    if sliding:
        one = put(to_bfloat16(np.ones(dim, dtype=np.float32)))
        runtime.dispatch("llmopt_rotary_attention_bf16", [b_rows, one, one, step, step, b_k, b_v, out],
                         u32s(m, heads, kv, dim, vdim, n, heads * vdim, capacity, span, 1, slots, 0) +
                         struct.pack("<ffff", scale, softcap, 1e-6, 1.0), *GRID)
        rows = b_rows.numpy(np.uint16).reshape(m, n)  # normed in place
    else:
        runtime.dispatch("llmopt_chunk_attention_bf16", [b_rows, put(sinks), step, b_k, b_v, out],
                         u32s(m, heads, kv, dim, vdim, capacity, span, slots, int(sink)) + struct.pack("<ff", scale, softcap),
                         *GRID)
    got = from_bfloat16(out.numpy(np.uint16)).reshape(m, heads, vdim).astype(np.float64)
    assert np.isfinite(got).all()

    wide = lambda a: from_bfloat16(a).astype(np.float64)
    q = wide(rows[:, :heads * dim]).reshape(m, heads, dim)
    fresh_k = wide(rows[:, heads * dim:heads * dim + kv * dim]).reshape(m, kv, dim)
    fresh_v = wide(rows[:, heads * dim + kv * dim:]).reshape(m, kv, vdim)
    begin = max(0, first - span)
    past = np.arange(begin, first) % capacity
    positions, seen_by = np.arange(begin, first + m), np.arange(first, first + m)
    gap = seen_by[:, None] - positions[None, :]
    visible = (gap >= 0) & ((gap < span) if sliding else (seen_by[:, None] // span == positions[None, :] // span))
    for head in range(heads):
        group = head // (heads // kv)
        keys = np.concatenate([wide(ring_k[slot, group])[past], fresh_k[:, group]])
        values = np.concatenate([wide(ring_v[slot, group])[past], fresh_v[:, group]])
        score = q[:, head] @ keys.T * scale
        if softcap:
            score = softcap * np.tanh(score / softcap)
        score = np.where(visible, score, -np.inf)
        top = np.maximum(score.max(axis=1), wide(sinks)[head] if sink and not sliding else -np.inf)
        weights = np.exp(score - top[:, None])
        total = weights.sum(axis=1) + (np.exp(wide(sinks)[head] - top) if sink and not sliding else 0.0)
        expected = weights @ values / total[:, None]
        error = np.abs(got[:, head] - expected)
        assert (error <= 2.0 ** -8 * np.abs(expected) + 2.0 ** -13 * np.abs(values).max()).all(), (head, error.max())


@pytest.mark.parametrize("m,heads,kv,dim,vdim,span,softcap,sink,first,sliding", [
    (513, 4, 2, 128, 128, 4096, 0.0, True, 0, False),         # one key more than eight stages
    (1100, 4, 1, 128, 128, 1500, 0.0, True, 1437, False),     # a chunk's end in the second tile
    (640, 2, 2, 128, 128, 700, 0.0, False, 2000, True),       # a window whose ring has turned
    (1001, 3, 3, 128, 128, 1007, 30.0, True, 940, False),     # bounded scores, stages across the ring's end
    (1025, 2, 1, 128, 128, 4096, 50.0, True, 63, False),
    (1061, 4, 2, 64, 64, 1040, 0.0, False, 1000, True),
    (1030, 6, 2, 64, 64, 2048, 0.0, True, 1, False),
    (660, 4, 2, 128, 128, 640, 0.0, True, 0, False),          # the last rows behind a chunk's end: one stage, a group without any
])
def test_groups_of_waves_in_turns(runtime, m, heads, kv, dim, vdim, span, softcap, sink, first, sliding):
    """Portions whose rows walk over many keys: 128 rows whose stages two groups of waves share."""
    test_tiles(runtime, m, heads, kv, dim, vdim, span, softcap, sink, first, sliding)


@pytest.mark.parametrize("m,dim,softcap", [(700, 128, 0.0), (1100, 128, 30.0), (1100, 128, 200.0), (1100, 64, 0.0)])
def test_infinite_values_behind_what_a_row_of_a_portion_sees(runtime, m, dim, softcap):
    """A weight of zero times an infinite value is NaN: not in rows none of whose 32 see any of its 32 keys."""
    rng = np.random.default_rng(m)
    heads, kv, span = 4, 2, 4096
    rows = to_bfloat16(rng.standard_normal((m, (heads + 2 * kv) * dim), dtype=np.float32))
    put = runtime.buffer_of_bytes
    zeros = np.zeros((1, kv, span, dim), dtype=np.uint16)

    def call():
        out = runtime.create_buffer(m * heads * dim * 2)
        runtime.dispatch("llmopt_chunk_attention_bf16", [put(rows), put(zeros), put(np.zeros(2, dtype=np.uint32)), put(zeros), put(zeros), out],
                         u32s(m, heads, kv, dim, dim, span, span, 1, 0) + struct.pack("<ff", dim ** -0.5, softcap), *GRID)
        return out.numpy(np.uint16).reshape(m, heads, dim)

    last = np.minimum(np.arange(m) // 32 * 32 + 31, m - 1)
    for bad, what in ((40, np.inf), (m - 70, -np.inf), (m - 1, np.nan)):
        column = (heads + kv + 1) * dim + 5
        rows[bad, column] = 0
        want = call()
        rows[bad, column] = to_bfloat16(np.array([what], dtype=np.float32))[0]
        got = call()
        rows[bad, column] = 0
        touched = np.zeros(got.shape, dtype=bool)
        touched[bad // 32 * 32 <= last, 2:, 5] = True
        assert (got[~touched] == want[~touched]).all(), (bad, what)
        assert not np.isfinite(from_bfloat16(got[bad:, 2:, 5])).any()


# rows, heads, kv_heads, dim, span, position of the first row: tiles in the order of their keys (several rounds of up to 64
# tiles, a chunk's end among them: 5, 16 and 64 tiles), more tiles than are ranked, one chunk, one round
@pytest.mark.parametrize("m,heads,kv,dim,span,first", [
    (300, 64, 8, 64, 512, 3000), (300, 64, 8, 128, 100, 37), (1024, 32, 8, 64, 700, 650), (4096, 8, 2, 32, 1000, 999),
    (4090, 16, 2, 32, 63, 5), (4100, 8, 2, 32, 1000, 7), (700, 64, 8, 64, 2048, 100), (200, 4, 2, 64, 64, 10)])
def test_float32_portions_over_the_ends_of_chunks(runtime, m, heads, kv, dim, span, first):
    """Against float64: sums of up to 1000 weights and 128 products in float32, and exponentials a few units off, move a
    weighted mean by less than 2^-15 of the largest value."""
    g = torch.Generator(device="cuda").manual_seed(m + heads)
    normal = lambda *shape: torch.randn(*shape, generator=g, device="cuda")
    rows, ring_k, ring_v = normal(m, (heads + 2 * kv) * dim), normal(kv, span, dim), normal(kv, span, dim)
    out, sinks = torch.full((m, heads, dim), float("nan"), device="cuda"), torch.zeros(heads, device="cuda").bfloat16()
    step = torch.tensor([first, 0], dtype=torch.int32, device="cuda")
    at = torch.arange(first, first + m, device="cuda")
    begin = first - first % span
    past = torch.arange(begin, first, device="cuda")
    places = torch.cat([past, at])
    seen = (places[None] <= at[:, None]) & (places[None] // span == at[:, None] // span)
    split = lambda a, h: a.double().view(m, h, dim)
    q, k, v = split(rows[:, :heads * dim], heads), split(rows[:, heads * dim:(heads + kv) * dim], kv), split(rows[:, (heads + kv) * dim:], kv)
    old_k, old_v = ring_k[:, past % span].double(), ring_v[:, past % span].double()
    torch.cuda.synchronize()
    wrap = lambda t: runtime.wrap(t.data_ptr(), t.numel() * t.element_size())
    runtime.dispatch("llmopt_chunk_attention_f32", [wrap(t) for t in (rows, sinks, step, ring_k, ring_v, out)],
                     u32s(m, heads, kv, dim, dim, span, span, 1, 0) + struct.pack("<ff", dim ** -0.5, 0.0), *GRID)
    for head in range(heads):
        group = head // (heads // kv)
        keys, values = torch.cat([old_k[group], k[:, group]]), torch.cat([old_v[group], v[:, group]])
        score = (q[:, head] @ keys.T * dim ** -0.5).masked_fill(~seen, float("-inf"))
        error = (out[:, head].double() - torch.softmax(score, dim=1) @ values).abs().max()
        assert error <= 2.0 ** -15 * values.abs().max(), (head, error)  # (a row that no tile wrote is NaN)


def test_portion_of_more_tiles_than_a_grid_has_rows(runtime):
    """64 * 65536 rows and a few: chunks of 64 stand alone, a thousand of them and the last ones against float64."""
    m, dim, span = 64 * 65536 + 70, 32, 64
    generator = torch.Generator(device="cuda").manual_seed(5)
    rows = torch.randn(m, 3 * dim, generator=generator, device="cuda", dtype=torch.bfloat16)
    step, sinks = torch.zeros(2, dtype=torch.int32, device="cuda"), torch.zeros(8, dtype=torch.bfloat16, device="cuda")
    keys, values = (torch.zeros(span, dim, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    out = torch.full((m, dim), float("nan"), dtype=torch.bfloat16, device="cuda")
    torch.cuda.synchronize()
    wrap = lambda t: runtime.wrap(t.data_ptr(), t.numel() * t.element_size())
    runtime.dispatch("llmopt_chunk_attention_bf16", [wrap(t) for t in (rows, sinks, step, keys, values, out)],
                     u32s(m, 1, 1, dim, dim, span, span, 1, 0) + struct.pack("<ff", dim ** -0.5, 0.0), *GRID)
    chunks = (m + span - 1) // span
    for chunk in [0, 1, *torch.linspace(2, chunks - 4, 1000).long().tolist(), chunks - 3, chunks - 2, chunks - 1]:
        part = rows[chunk * span:(chunk + 1) * span].double()
        q, k, v = part[:, :dim], part[:, dim:2 * dim], part[:, 2 * dim:]
        seen = torch.ones(len(part), len(part), dtype=torch.bool, device="cuda").tril()
        expected = torch.softmax((q @ k.T * dim ** -0.5).masked_fill(~seen, float("-inf")), dim=1) @ v
        error = (out[chunk * span:(chunk + 1) * span].double() - expected).abs()
        assert (error <= 2.0 ** -8 * expected.abs() + 2.0 ** -13 * v.abs().max()).all(), (chunk, error.max())
