"""A prompt of the gated delta rule in one portion against the same in portions of whole chunks: enough chunks and heads
for three workgroups a compute unit against few enough for two, and every width of the outputs' tiles.  Chunk borders are
the same, so the two differ by the order in which the decays' low-rank products are summed (a few times 2^-24) and the
rounding of an output to bfloat16 that this can move: one unit, 2^-8 of the value.  And one portion of as many
workgroups against the rule token by token in float64."""
import struct

import numpy as np
import pytest

from llmopt_amd.safetensors_file import from_bfloat16, to_bfloat16
from oracle import hybrid_model, parallel_model
from tests.gpu_util import u32s

pytestmark = pytest.mark.gpu
GRID = ((1, 1, 1), (256, 1, 1))


@pytest.fixture(scope="module")
def runtime():
    from llmopt_amd.native import Runtime
    rt = Runtime()
    yield rt
    rt.close()


TAPS, RANKS = 4, (8, 16)
EPSILON, OUT_SCALE = 1e-6, 0.5


def make_inputs(m, heads, kv_heads, dim, vdim, kind):
    """Rows as the joint input leaves them, the columns of their parts, write strengths and weights."""
    rng = np.random.default_rng(m + dim)
    n_out = heads * vdim
    channels = 2 * kv_heads * dim + n_out
    decay_at = (channels + 7) // 8 * 8
    gate_at, ld = decay_at + RANKS[0], decay_at + RANKS[0] + RANKS[1]
    store = to_bfloat16 if kind == "bf16" else (lambda a: a)
    rows = store(rng.standard_normal((m, ld), dtype=np.float32))
    beta = rng.standard_normal((m, heads), dtype=np.float32)
    bf16 = lambda *shape, gain=1.0: to_bfloat16(rng.standard_normal(shape, dtype=np.float32) * np.float32(gain))
    weights = [bf16(heads * dim, RANKS[0], gain=RANKS[0] ** -0.5), bf16(heads * dim), bf16(heads, gain=0.5),
               bf16(n_out, RANKS[1], gain=RANKS[1] ** -0.5), bf16(vdim), bf16(channels, TAPS)]
    return rows, (decay_at, gate_at), beta, weights


def run_portions(runtime, portions, sizes, kind, rows, columns, beta, weights):
    heads, kv_heads, dim, vdim = sizes
    put, n_out, ld = runtime.buffer_of_bytes, heads * vdim, rows.shape[1]
    weights, channels = [put(w) for w in weights], 2 * kv_heads * dim + n_out
    ring, state = runtime.create_buffer(TAPS * channels * 4), put(np.zeros((heads, dim, vdim), dtype=np.float32))
    out, at = [], 0
    for count in portions:
        target = put(np.zeros((count, n_out), dtype=rows.dtype))
        runtime.dispatch(f"llmopt_gated_delta_{kind}",
                         [put(rows[at:at + count]), put(beta[at:at + count]), *weights, ring, state,
                          put(np.array([at, 0], dtype=np.uint32)), target],
                         u32s(count, heads, kv_heads, dim, vdim, TAPS, 1, ld, 0, *columns, ld, *RANKS, n_out, 0) +
                         struct.pack("<ff", EPSILON, OUT_SCALE), *GRID)
        part = target.numpy(rows.dtype)
        out.append((from_bfloat16(part) if kind == "bf16" else part).reshape(count, n_out))
        at += count
    return np.concatenate(out), state.numpy(np.float32, (heads, dim, vdim))


@pytest.mark.parametrize("m,heads,kv_heads,dim,vdim", [
    (2115, 16, 4, 128, 128), (2070, 16, 16, 72, 40), (2049, 20, 5, 128, 200), (200, 4, 2, 256, 120), (130, 2, 1, 64, 72)])
@pytest.mark.parametrize("kind", ["bf16", "f32"])
def test_one_portion_is_several(runtime, m, heads, kv_heads, dim, vdim, kind):
    inputs = make_inputs(m, heads, kv_heads, dim, vdim, kind)
    (whole, whole_state), (parts, parts_state) = (
        run_portions(runtime, portions, (heads, kv_heads, dim, vdim), kind, *inputs)
        for portions in ([m], [640] * (m // 640) + [m % 640] if m > 640 else [64, m - 64]))
    assert np.isfinite(whole).all() and np.abs(whole).max() > 0
    unit = 2.0 ** -8 if kind == "bf16" else 2.0 ** -14
    assert (np.abs(whole - parts) <= unit * np.abs(whole) + 2.0 ** -14 * np.abs(whole).max()).all()
    assert np.abs(whole_state - parts_state).max() <= 2.0 ** -14 * np.abs(whole_state).max()


def exact_rule(sizes, rows, columns, beta, weights):
    """Outputs [m, heads * vdim] and the state behind the last token, float64."""
    heads, kv_heads, dim, vdim = sizes
    m, (decay_at, gate_at) = rows.shape[0], columns
    w_decay, dt_bias, a_log, w_gate, norm, conv = (from_bfloat16(w).astype(np.float64) for w in weights)
    rows = (from_bfloat16(rows) if rows.dtype != np.float32 else rows).astype(np.float64)
    key_columns = kv_heads * dim
    mixed = hybrid_model.silu(parallel_model.short_conv(rows[:, :2 * key_columns + heads * vdim], conv))
    q = parallel_model.unit(mixed[:, :key_columns].reshape(m, kv_heads, dim)) / np.sqrt(dim)
    k = parallel_model.unit(mixed[:, key_columns:2 * key_columns].reshape(m, kv_heads, dim))
    q, k = (np.repeat(a, heads // kv_heads, axis=1) for a in (q, k))
    v = mixed[:, 2 * key_columns:].reshape(m, heads, vdim)
    step = hybrid_model.softplus(rows[:, decay_at:decay_at + RANKS[0]] @ w_decay.T + dt_bias).reshape(m, heads, dim)
    decay, beta = np.exp(-np.exp(a_log)[None, :, None] * step), hybrid_model.sigmoid(beta.astype(np.float64))
    state, out = np.zeros((heads, dim, vdim)), np.zeros((m, heads, vdim))
    for i in range(m):
        state *= decay[i][:, :, None]
        u = beta[i][:, None] * (v[i] - (state * k[i][:, :, None]).sum(axis=1))
        state += k[i][:, :, None] * u[:, None, :]
        out[i] = (state * q[i][:, :, None]).sum(axis=1)
    gate = hybrid_model.sigmoid(rows[:, gate_at:gate_at + RANKS[1]] @ w_gate.T).reshape(m, heads, vdim)
    return (hybrid_model.rms_unit(out, EPSILON) * norm * gate * OUT_SCALE).reshape(m, -1), state


@pytest.mark.parametrize("m,heads,kv_heads,dim,vdim", [(130, 176, 88, 72, 24), (65, 300, 100, 128, 40), (192, 180, 180, 100, 16)])
@pytest.mark.parametrize("kind", ["bf16", "f32"])
def test_three_workgroups_against_float64(runtime, m, heads, kv_heads, dim, vdim, kind):
    """As many chunks and heads as take three workgroups a compute unit.  float32: the bound of the restatement's rows.
    bfloat16: v, the gate in front of its sigmoid and the output are rounded, 2^-9 of each value at most."""
    sizes, inputs = (heads, kv_heads, dim, vdim), make_inputs(m, heads, kv_heads, dim, vdim, kind)
    actual, expected = run_portions(runtime, [m], sizes, kind, *inputs), exact_rule(sizes, *inputs)
    for got, true in zip(actual, expected):
        error = np.linalg.norm((got - true).reshape(-1)) / np.linalg.norm(true.reshape(-1))
        print(kind, sizes, error, flush=True)
        assert error <= (2.0 ** -7 if kind == "bf16" else 3e-5)
