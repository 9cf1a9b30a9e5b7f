"""Performance cases: what programs built on this package have it do, from one small linear call to whole prompts.

`listed()` and `draw()` give cases, `prepare()` what a program holds before the call, `run()` one pass through the
public entry points, `exact()` the same outputs in plain float64 torch.  Sizes are those of the repository's own
benchmark and test configurations and generic ones around them.
"""
from __future__ import annotations

import math
import struct

import numpy as np
import torch

import llmopt_amd.torch_ops  # noqa: F401  (registers torch.ops.llmopt.w4a16_linear)
from llmopt_amd.decode_step import DecodeConfig, DecodeStep
from llmopt_amd.layered_model import LayeredConfig, LayeredModel
from llmopt_amd.native import DispatchList, Prebaked, Runtime
from llmopt_amd.w4a16_model import W4a16Model

GROUP = 64
EPSILON = 1e-5

# The 30-layer transformer of the decode-step benchmark, and a wider one with heads of 128.
SMALL = dict(hidden=576, q_heads=9, kv_heads=3, head_dim=64, mlp=1536, layers=30, vocabulary=49152)
WIDE = dict(hidden=2048, q_heads=16, kv_heads=4, head_dim=128, mlp=8192, layers=4, vocabulary=32768)
# A recurrent layer with a dense feed-forward and an attention layer with routed experts.
BAROVIK = dict(design="Barovik", width=2048, heads=32, kv_heads=8, dim=128, span=2048, state_heads=64, state=128, ff=8192,
               experts=16, top=4, expert_ff=1024, shared_ff=1024, pairs=1, vocabulary=32768)
BAROVIK_SMALL = dict(design="Barovik", width=1024, heads=16, kv_heads=4, dim=64, span=2048, state_heads=32, state=128, ff=4096,
                     experts=16, top=4, expert_ff=512, shared_ff=1024, pairs=2, vocabulary=32768)
# Window attention and the gated delta rule side by side.
KOKETAR = dict(design="Koketar", width=2048, heads=16, kv_heads=4, dim=128, span=2048, state_heads=16, state=128, ff=8192,
               pairs=2, vocabulary=32768)
KOKETAR_SMALL = dict(design="Koketar", width=1024, heads=16, kv_heads=4, dim=64, span=2048, state_heads=8, state=128, ff=4096,
                     pairs=4, vocabulary=32768)
RANK = 128  # of Koketar's low-rank products


def listed():
    return [
        # One projection of one token of a small model: the smallest call, through the torch operator.
        dict(name="linear of one token", kind="linear", m=1, k=576, n=1536, bias=False),
        # A wide model's projection for the tokens of a batch of sequences (or a few drafted tokens).
        dict(name="linear of a batch", kind="linear", m=24, k=4096, n=14336, bias=True),
        # The same for a whole prompt.
        dict(name="linear of a prompt", kind="linear", m=2048, k=4096, n=14336, bias=False),
        # Decode attention of one layer: a serving batch with contexts of very different lengths over the Q8 cache.
        dict(name="decode attention", kind="cache_attention", batch=16, heads=32, kv_heads=8, dim=128, shortest=512,
             longest=8192, paged=False),
        # Attention of one layer over a long prompt.
        dict(name="prompt attention", kind="prompt_attention", heads=32, kv_heads=8, dim=128, tokens=4096),
        # The quantised transformer as served: a prompt, the next token of one sequence, of a batch of sequences.
        dict(name="transformer prompt", kind="w4_prompt", tokens=700, **SMALL),
        dict(name="transformer token", kind="w4_token", context=2048, **SMALL),
        dict(name="transformer batch", kind="w4_batch", batch=32, shortest=1024, longest=2048, **SMALL),
        # Layered decoders: a long prompt, and a short prompt with the tokens of a reply behind it.
        dict(name="recurrent and routed prompt", kind="layered_prompt", tokens=2048, **BAROVIK),
        dict(name="recurrent and routed reply", kind="layered_reply", tokens=64, reply=24, **BAROVIK_SMALL),
        dict(name="side by side prompt", kind="layered_prompt", tokens=3001, **KOKETAR),
        dict(name="side by side reply", kind="layered_reply", tokens=64, reply=24, **KOKETAR_SMALL),
    ]


def _log(rng, low, high):
    """A whole number, its logarithm uniform."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _draw_linear(rng):
    m, k, n = _log(rng, 1, 2048), GROUP * _log(rng, 8, 224), _log(rng, 256, 14336)
    if rng.random() < 0.5:
        n = max(256, n // 64 * 64)
    while m * k * n > 2048 * 4096 * 14336:
        m = (m + 1) // 2
    return dict(kind="linear", m=m, k=k, n=n, bias=rng.random() < 0.5)


def _draw_cache_attention(rng):
    heads, kv_heads, dim = rng.choice([(32, 8, 128), (32, 8, 128), (16, 4, 64), (9, 3, 64), (16, 16, 64), (16, 4, 256)])
    longest = _log(rng, 100, 8192)
    batch = min(_log(rng, 1, 64), max(1, 16 * 8192 * 8 * 128 // (longest * kv_heads * dim)))
    return dict(kind="cache_attention", batch=batch, heads=heads, kv_heads=kv_heads, dim=dim,
                shortest=max(1, longest // _log(rng, 1, 16)), longest=longest, paged=rng.random() < 0.5)


def _draw_prompt_attention(rng):
    heads, kv_heads, dim = rng.choice([(32, 8, 128), (16, 4, 128), (16, 4, 64), (9, 3, 64), (16, 8, 256)])
    return dict(kind="prompt_attention", heads=heads, kv_heads=kv_heads, dim=dim, tokens=_log(rng, 60, 4096 if dim < 256 else 2048))


def _draw_transformer(rng):
    shape = dict(rng.choice([SMALL, SMALL, WIDE]))
    kind = rng.choice(["w4_prompt", "w4_token", "w4_batch"])
    if kind == "w4_prompt":
        return dict(kind=kind, tokens=_log(rng, 20, 2048), **shape)
    if kind == "w4_token":
        return dict(kind=kind, context=_log(rng, 20, 2048), **shape)
    longest = _log(rng, 100, 2048)
    return dict(kind=kind, batch=_log(rng, 2, 48), shortest=max(64, longest // 4), longest=longest, **shape)


def _draw_layered(rng):
    shape = dict(rng.choice([BAROVIK, BAROVIK_SMALL, KOKETAR, KOKETAR_SMALL]))
    shape["span"] = rng.choice([512, 1024, 2048])
    if rng.random() < 0.5:
        return dict(kind="layered_prompt", tokens=_log(rng, 30, 3001), **shape)
    return dict(kind="layered_reply", tokens=_log(rng, 16, 256), reply=rng.randint(8, 24), **shape)


def draw(rng):
    return rng.choice([_draw_linear, _draw_linear, _draw_cache_attention, _draw_prompt_attention, _draw_transformer,
                       _draw_transformer, _draw_layered, _draw_layered])(rng)


# ---- what a program holds before the call -----------------------------------------------------------------

_runtimes: dict = {}


def _runtime(kind) -> Runtime:
    """Two runtimes: one whose launches go to torch's stream (single operators on tensors), one with a stream of its
    own, on which models capture their plans."""
    if kind not in _runtimes:
        _runtimes[kind] = Runtime()
        if kind == "tensors":
            _runtimes[kind].set_stream(torch.cuda.current_stream().cuda_stream)
    return _runtimes[kind]


def _wrap(runtime, tensor):
    return runtime.wrap(tensor.data_ptr(), tensor.numel() * tensor.element_size())


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape, gain=1.0, dtype=torch.float16):
    return (torch.randn(*shape, generator=g, device="cuda") * gain).to(dtype)


def _uniform(g, low, high, *shape, dtype=torch.float16):
    return (torch.rand(*shape, generator=g, device="cuda") * (high - low) + low).to(dtype)


def _whole(g, low, high, *shape, dtype=torch.int64):
    """Whole numbers from low to high - 1."""
    return torch.randint(low, high, shape, generator=g, device="cuda").to(dtype)


def _w4(g, n, k):
    """Packed nibbles [n, k / 2] and group scales [n, k / 64], as a checkpoint holds them."""
    return _whole(g, 0, 256, n, k // 2, dtype=torch.uint8), _uniform(g, 0.005, 0.02, n, k // GROUP)


def _linear_inputs(case, seed):
    g, m, n, k = _generator(seed), case["m"], case["n"], case["k"]
    return _normal(g, m, k), *_w4(g, n, k), _normal(g, n) if case["bias"] else None


def _pool(g, tokens, elements):
    """Cache slots: int8 values as the quantiser leaves normal ones, then a scale for every 64."""
    values = torch.clamp(torch.round(torch.randn(tokens, elements, generator=g, device="cuda") * 38.0), -127, 127).to(torch.int8)
    scales = _uniform(g, 0.02, 0.035, tokens, elements // GROUP)
    return torch.cat([values.view(torch.uint8), scales.view(torch.uint8).view(tokens, -1)], dim=1).contiguous()


def _cache_inputs(case, seed):
    g, batch, kv, dim = _generator(seed), case["batch"], case["kv_heads"], case["dim"]
    lengths = _whole(g, case["shortest"], case["longest"] + 1, batch, dtype=torch.int32)
    total = int(lengths.sum())
    slots = torch.arange(total, device="cuda")
    if case["paged"]:  # pages of 16 tokens anywhere in the pool
        pages = (total + 15) // 16
        slots = torch.randperm(pages, generator=g, device="cuda")[slots // 16] * 16 + slots % 16
        total = pages * 16
    offsets = (torch.cumsum(lengths, 0) - lengths).to(torch.int32)
    return dict(query=_normal(g, batch, case["heads"], 1, dim), key=_normal(g, batch, kv, 1, dim),
                value=_normal(g, batch, kv, 1, dim), pool=_pool(g, total, 2 * kv * dim), slots=slots.to(torch.int32),
                lengths=lengths, offsets=offsets)


def _prompt_attention_inputs(case, seed):
    g, t, dim = _generator(seed), case["tokens"], case["dim"]
    return tuple(_normal(g, 1, case[heads], t, dim) for heads in ("heads", "kv_heads", "kv_heads"))


def _transformer_config(case):
    return DecodeConfig(hidden=case["hidden"], q_heads=case["q_heads"], kv_heads=case["kv_heads"], head_dim=case["head_dim"],
                        mlp=case["mlp"], layers=case["layers"], vocabulary=case["vocabulary"], epsilon=EPSILON)


def _transformer_weights(case, g):
    h, q, kv, mlp = case["hidden"], case["q_heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"], case["mlp"]
    shapes = dict(q=(q, h), k=(kv, h), v=(kv, h), o=(h, q), gate=(mlp, h), up=(mlp, h), down=(h, mlp))
    layers = [dict(attn_norm=_uniform(g, 0.5, 1.5, h), ffn_norm=_uniform(g, 0.5, 1.5, h),
                   **{name: _w4(g, *shape) for name, shape in shapes.items()}) for _ in range(case["layers"])]
    return dict(embedding=_normal(g, case["vocabulary"], h, gain=0.5), layers=layers, final_norm=_uniform(g, 0.5, 1.5, h),
                lm_head=_w4(g, case["vocabulary"], h))


def _device_weights(runtime, weights):
    put = lambda value: tuple(_wrap(runtime, t) for t in value) if isinstance(value, tuple) else _wrap(runtime, value)
    return dict(embedding=put(weights["embedding"]), final_norm=put(weights["final_norm"]), lm_head=put(weights["lm_head"]),
                layers=[{name: put(value) for name, value in layer.items()} for layer in weights["layers"]])


def _batch_inputs(case, g, config):
    """Contexts of a batch in one pool, with room for every sequence's next token."""
    batch = case["batch"]
    lengths = _whole(g, case["shortest"], case["longest"] + 1, batch)
    starts = torch.cumsum(lengths + 1, 0) - (lengths + 1)
    total = int((lengths + 1).sum())
    pool = _pool(g, total, config.token_elements)
    return pool, lengths, starts, total, _whole(g, 0, case["vocabulary"], batch)


def _layered_config(case):
    head = dict(heads=case["heads"], kv_heads=case["kv_heads"], dim=case["dim"], vdim=case["dim"], scale=case["dim"] ** -0.5,
                mask={"size": case["span"]})
    config = dict(architecture=case["design"], vocab=case["vocabulary"], width=case["width"], norm={"eps": 1e-6})
    if case["design"] == "Barovik":
        mamba = dict(type="mamba2", mlp=dict(kind="dense", ff=case["ff"]),
                     mixer=dict(heads=case["state_heads"], vdim=64, state=case["state"], groups=1, conv=4, norm_groups=1))
        attention = dict(type="attention", mixer=dict(**head, softcap=30.0, v_mix=True),
                         mlp=dict(kind="moe", router=dict(experts=case["experts"], top=case["top"]),
                                  expert=dict(ff=case["expert_ff"]), shared=dict(ff=case["shared_ff"])))
        return dict(config, embedding={"scale": 1.0}, layers=[mamba, attention] * case["pairs"])
    left = dict(head, rot={"base": 1e6, "dims": case["dim"], "scaling": {"factor": 4.0}})
    right = dict(heads=case["state_heads"], kv_heads=case["state_heads"], dim=case["state"], vdim=case["state"], conv=4)
    layer = dict(type="parallel", mlp=dict(kind="dense", ff=case["ff"], limit=7.0),
                 mixer=dict(left=left, right=right, left_scale=0.5, right_scale=0.5))
    return dict(config, residual_mult=0.5, logit_softcap=30.0, layers=[layer] * case["pairs"])


def _layered_weights(case, seed):
    """bfloat16 tensors under the names of a weight file: projections that keep the scale of their input."""
    g, out = _generator(seed), {}
    parsed = LayeredConfig.parse(_layered_config(case))
    for name, shape in parsed.tensor_shapes().items():
        shape = tuple(RANK if size is None else size for size in shape)
        kind = name.rsplit(".", 1)[-1]
        if "norm" in kind:
            around_zero = case["design"] == "Koketar" and ".mix." not in name
            value = _uniform(g, -0.5 if around_zero else 0.5, 0.5 if around_zero else 1.5, *shape, dtype=torch.bfloat16)
        elif kind in ("A_log", "dt_bias", "D", "b", "sink") and len(shape) < 2:
            value = _uniform(g, -1.0, 1.0, *shape, dtype=torch.bfloat16)
        elif kind == "vmix":
            value = _uniform(g, 0.2, 0.8, 1, dtype=torch.bfloat16).reshape(())
        else:
            value = _normal(g, *shape, gain=0.5 if name == "embed" else shape[-1] ** -0.5, dtype=torch.bfloat16)
        out[name] = value
    return parsed, out


def _tokens(case, seed, count):
    return np.random.default_rng([int(seed), 7]).integers(0, case["vocabulary"], count)


def _prepare_transformer(case, seed):
    runtime, g, config = _runtime("models"), _generator(seed), _transformer_config(case)
    weights = _transformer_weights(case, g)
    torch.cuda.synchronize()
    device = _device_weights(runtime, weights)
    state = dict(case=case, weights=weights)  # (the tensors own the memory)
    if case["kind"] == "w4_batch":
        pool, lengths, starts, total, tokens = _batch_inputs(case, g, config)
        lengths, starts, tokens = (t.cpu().numpy() for t in (lengths, starts, tokens))
        torch.cuda.synchronize()
        step = DecodeStep(runtime, config, {}, case["batch"], _wrap(runtime, pool),
                          runtime.buffer_of_bytes(np.arange(total, dtype=np.uint32)), starts, lengths, starts + lengths, lengths,
                          device_weights=device)
        logits = torch.zeros(case["batch"], case["vocabulary"], dtype=torch.float16, device="cuda")
        name, buffers, parameters, grid, group = step.dispatches[-1]
        step.dispatches[-1] = ("llmopt_w4a16_lm_head_argmax_extra_f16", buffers + [_wrap(runtime, logits)], parameters, grid, group)
        step.tokens.write(tokens.astype(np.int64))
        torch.cuda.synchronize()
        plan = Prebaked(runtime, step.dispatches, step.tokens, step.token_ids)
        return dict(state, pool=pool, step=step, plan=plan, first=int(tokens[0]), past=int(lengths[0]), logits=logits)
    count = case["tokens"] if case["kind"] == "w4_prompt" else case["context"]
    model = W4a16Model(runtime, config, device, slots=1, max_context=count + 64)
    tokens = _tokens(case, seed, count + 1)
    state.update(model=model, tokens=tokens[:count].tolist())
    if case["kind"] == "w4_token":
        sequence = model.open()
        model.step(sequence, state["tokens"])
        model.decode(sequence, int(tokens[count]))
        state.update(sequence=sequence, token=int(tokens[count]))
    return state


def _prepare_layered(case, seed):
    parsed, tensors = _layered_weights(case, seed)
    patterns = {name: t.view(torch.int16).cpu().numpy().view(np.uint16) for name, t in tensors.items()}
    model = LayeredModel(_runtime("models"), parsed, patterns, slots=2, max_context=16384)
    tokens = _tokens(case, seed, case["tokens"] + case.get("reply", 0))
    state = dict(case=case, model=model, tokens=tokens[:case["tokens"]].tolist(), reply=tokens[case["tokens"]:].tolist())
    if state["reply"]:
        model.decode_plan()
    return state


def prepare(case, seed):
    kind = case["kind"]
    if kind == "linear":
        return dict(case=case, inputs=_linear_inputs(case, seed))
    if kind.startswith("w4"):
        return _prepare_transformer(case, seed)
    if kind.startswith("layered"):
        return _prepare_layered(case, seed)
    runtime = _runtime("tensors")
    if kind == "cache_attention":
        c = _cache_inputs(case, seed)
        batch, heads, kv, dim = case["batch"], case["heads"], case["kv_heads"], case["dim"]
        elements = 2 * kv * dim
        out = torch.zeros(batch, 1, heads, dim, dtype=torch.float16, device="cuda")
        parameters = struct.pack("<12If4I", batch, heads, kv, 0, dim, 0, 0, elements, 0, kv * dim, GROUP,
                                 elements + 2 * (elements // GROUP), dim ** -0.5, 1, 0, 0, int(c["lengths"].max()))
        tensors = [c["query"], c["key"], c["value"], c["pool"], c["slots"], c["slots"], out, c["lengths"], c["offsets"]]
        name = "llmopt_attention_q8_paged_batched"
    else:
        tokens, heads, dim = case["tokens"], case["heads"], case["dim"]
        query, key, value = _prompt_attention_inputs(case, seed)
        out = torch.zeros(tokens, heads, dim, dtype=torch.float16, device="cuda")
        parameters = struct.pack("<8If5I", 1, heads, tokens, tokens, dim, 0, 0, 1, dim ** -0.5, case["kv_heads"], 1, 0, 0, 0)
        tensors = [query, key, value, query, out]
        name = f"llmopt_attention_f16_simd_h{dim}"
    buffers = [_wrap(runtime, t) for t in tensors]
    calls = DispatchList([(name, buffers, parameters, (out.numel() // 64 * 32, 1, 1), (256, 1, 1))])
    return dict(case=case, tensors=tensors, calls=calls, out=out)


# ---- one pass ---------------------------------------------------------------------------------------------

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        return torch.ops.llmopt.w4a16_linear(*state["inputs"])
    if kind in ("cache_attention", "prompt_attention"):
        batch = _runtime("tensors").begin_batch()
        batch.dispatch_all(state["calls"])
        batch.commit_async()
        return state["out"]
    if kind == "w4_batch":
        state["plan"].execute(state["first"], state["past"])
        return {"logits": state["logits"]}
    model = state["model"]
    if kind == "w4_token":
        sequence = state["sequence"]
        sequence.position = case["context"]  # the same token again: its cache slot is written anew
        model.decode(sequence, state["token"])
        return {"logits": model.logits_row()}
    sequence = model.open()
    if kind in ("w4_prompt", "layered_prompt"):
        logits = model.step(sequence, state["tokens"], [len(state["tokens"]) - 1])
    else:
        model.step(sequence, state["tokens"])
        for token in state["reply"]:
            model.decode(sequence, token)
        logits = model.logits_row()
    model.close(sequence)
    return {"logits": logits}


# ---- what a pass cannot do without ------------------------------------------------------------------------

def _w4_bytes(n, k):
    return n * k // 2 + 2 * n * (k // GROUP)


def _transformer_work(case):
    h, q, kv, mlp, layers = (case["hidden"], case["q_heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"], case["mlp"],
                             case["layers"])
    matrices = [(q, h), (kv, h), (kv, h), (h, q), (mlp, h), (mlp, h), (h, mlp)]
    stride = layers * (2 * kv + 2 * (2 * kv // GROUP))
    weights = layers * sum(_w4_bytes(*m) for m in matrices) + _w4_bytes(case["vocabulary"], h)
    per_token, head = layers * 2 * sum(n * k for n, k in matrices), 2 * h * case["vocabulary"]
    rows = case.get("batch", 1)
    moved = weights + rows * 2 * case["vocabulary"]
    if case["kind"] == "w4_prompt":
        t = case["tokens"]
        return dict(bytes=moved + t * (stride + 2 * h), flops=t * per_token + head + layers * 2 * q * t * (t + 1))
    contexts = case["context"] if case["kind"] == "w4_token" else rows * (case["shortest"] + case["longest"]) // 2
    return dict(bytes=moved + contexts * stride, flops=rows * (per_token + head) + layers * 4 * q * contexts)


def _layered_work(case):
    w, span, t, reply = case["width"], case["span"], case["tokens"], case.get("reply", 0)
    inner, rows = case["heads"] * case["dim"], case["kv_heads"] * case["dim"]
    if case["design"] == "Barovik":
        state_inner = case["state_heads"] * 64
        mixers = w * (3 * state_inner + 2 * case["state"] + case["state_heads"]) + w * (2 * inner + 2 * rows)
        used = 3 * w * (case["ff"] + case["top"] * case["expert_ff"] + case["shared_ff"]) + w * (case["experts"] + 1)
        held = used + 3 * w * (case["experts"] - case["top"]) * case["expert_ff"]
        keys = sum(n * (n + 1) / 2 for n in [span] * (t // span) + [t % span])
        state, scan = state_inner * case["state"], 6.0 * state_inner * case["state"]
    else:
        state_inner = case["state_heads"] * case["state"]
        mixers = w * (2 * inner + 2 * rows + 4 * state_inner + case["state_heads"] + 2 * RANK) + 2 * RANK * state_inner
        used = held = 3 * w * case["ff"]
        window = min(span, t)
        keys = window * (window + 1) / 2 + (t - window) * window
        state, scan = state_inner * case["state"], 8.0 * state_inner * case["state"]
    heads = w * case["vocabulary"]
    pairs = case["pairs"]
    flops = t * pairs * (2.0 * (mixers + used) + scan) + pairs * 4.0 * inner * keys
    moved = 2 * pairs * (mixers + held) + pairs * 8 * state + 2 * t * w
    if not reply:
        return dict(bytes=moved + 2 * heads + 4 * case["vocabulary"], flops=flops + 2.0 * heads)
    read = 2 * pairs * (mixers + used) + 2 * heads + pairs * (8 * state + 4 * rows * min(t, span))
    return dict(bytes=moved + reply * read, flops=flops + reply * (pairs * (2.0 * (mixers + used) + scan) + 2.0 * heads))


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        return dict(bytes=_w4_bytes(n, k) + 2 * m * (k + n) + (2 * n if case["bias"] else 0), flops=2 * m * n * k)
    if kind == "cache_attention":
        tokens, inner = case["batch"] * (case["shortest"] + case["longest"]) // 2, case["kv_heads"] * case["dim"]
        rows = case["heads"] * case["dim"]
        return dict(bytes=tokens * (2 * inner + 4 * inner // GROUP) + 4 * case["batch"] * rows, flops=4 * tokens * rows)
    if kind == "prompt_attention":
        t, rows = case["tokens"], case["heads"] * case["dim"]
        return dict(bytes=4 * t * (rows + case["kv_heads"] * case["dim"]), flops=2 * rows * t * (t + 1))
    return _transformer_work(case) if kind.startswith("w4") else _layered_work(case)


def tolerance(case):
    """About four times what the code was off from float64 when this was written: single operators 2 to 2.8e-4 (half
    precision results), transformer logits 2 to 6.5e-4, layered decoders' logits 1.7 to 5e-3 (bfloat16 operands); more
    where a router's close call may go the other way for a token."""
    kind = case["kind"]
    if kind in ("linear", "cache_attention", "prompt_attention"):
        return {"rel": 1.1e-3}
    if kind.startswith("w4"):
        return {"rel": 2.5e-3}
    return {"rel": 0.02 if case["design"] == "Koketar" else 0.03}


# ---- the same outputs in float64 --------------------------------------------------------------------------

def _f64(t):
    return t.to(torch.float64)


def _w4_f64(pair):
    """Low nibble first, two's complement, a scale for every 64 columns."""
    packed, scale = pair
    q = torch.stack([packed & 15, packed >> 4], dim=-1).reshape(packed.shape[0], -1).to(torch.int16)
    q = torch.where(q >= 8, q - 16, q)
    return _f64(q) * _f64(scale).repeat_interleave(GROUP, dim=1)


def _rms(x, weight, eps):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps) * _f64(weight)


def _silu(x):
    return x * torch.sigmoid(x)


def _attend(q, k, v, scale, seen, cap=0.0, sink=None):
    """q [t, H, d], k [s, G, d], v [s, G, e], seen [t, s] -> [t, H, e]."""
    per = q.shape[1] // k.shape[1]
    out = []
    for h in range(q.shape[1]):
        s = q[:, h] @ k[:, h // per].T * scale
        s = cap * torch.tanh(s / cap) if cap else s
        s = s.masked_fill(~seen, -math.inf)
        top = s.max(-1, keepdim=True).values
        e = torch.exp(s - top)
        total = e.sum(-1, keepdim=True)
        if sink is not None:
            total = total + torch.exp(sink[h] - top)
        out.append(e / total @ v[:, h // per])
    return torch.stack(out, dim=1)


def _places(t):
    return torch.arange(t, device="cuda")


def _unpacked(pool, elements):
    """Cache slots as float64 values."""
    q = _f64(pool[:, :elements].contiguous().view(torch.int8))
    return q * _f64(pool[:, elements:].contiguous().view(torch.float16)).repeat_interleave(GROUP, dim=1)


def _exact_cache_attention(case, seed):
    c, kv, dim = _cache_inputs(case, seed), case["kv_heads"], case["dim"]
    out = []
    for b in range(case["batch"]):
        start, length = int(c["offsets"][b]), int(c["lengths"][b])
        rows = _unpacked(c["pool"][c["slots"][start:start + length].long()], 2 * kv * dim).view(length, 2, kv, dim)
        k = torch.cat([rows[:, 0], _f64(c["key"][b]).transpose(0, 1)])
        v = torch.cat([rows[:, 1], _f64(c["value"][b]).transpose(0, 1)])
        seen = torch.ones(1, length + 1, dtype=torch.bool, device="cuda")
        out.append(_attend(_f64(c["query"][b]).transpose(0, 1), k, v, dim ** -0.5, seen))
    return torch.stack(out)


def _exact_prompt_attention(case, seed):
    q, k, v = (_f64(t[0]).transpose(0, 1) for t in _prompt_attention_inputs(case, seed))
    at = _places(case["tokens"])
    return _attend(q, k, v, case["dim"] ** -0.5, at[None, :] <= at[:, None])


def _rotated(x, positions):
    """Halves of a head turned by tables in half precision, as the package's interface hands them over."""
    d = x.shape[-1]
    frequency = (10000.0 ** (-np.arange(0, d, 2, dtype=np.float64) / d)).astype(np.float32)
    angle = (frequency[None, :] * np.asarray(positions, dtype=np.float32)[:, None]).astype(np.float32).astype(np.float64)
    cos, sin = (torch.from_numpy(f(angle).astype(np.float32).astype(np.float16)).cuda().double()[:, None] for f in (np.cos, np.sin))
    a, b = x[..., :d // 2], x[..., d // 2:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)


def _quantised(x):
    """Values as they come back from the cache: a half scale for every 64, whole numbers up to 127."""
    groups = x.reshape(*x.shape[:-1], -1, GROUP)
    scale = _f64((groups.abs().amax(-1, keepdim=True) / 127).to(torch.float16))
    scale = torch.where(scale == 0, torch.ones_like(scale), scale)
    return (torch.clamp(torch.round(groups / scale), -127, 127) * scale).reshape(x.shape)


def _transformer_layers(case, weights, x, positions, attend):
    """The residual stream behind the layers; attend(index, q, k, v) gives every row's attention."""
    t, dim = x.shape[0], case["head_dim"]
    for index, layer in enumerate(weights["layers"]):
        w = {name: _w4_f64(value) for name, value in layer.items() if isinstance(value, tuple)}
        h = _rms(x, layer["attn_norm"], EPSILON)
        q, k, v = ((h @ w[name].T).view(t, -1, dim) for name in "qkv")
        x = x + attend(index, _rotated(q, positions), _rotated(k, positions), v).reshape(t, -1) @ w["o"].T
        h = _rms(x, layer["ffn_norm"], EPSILON)
        x = x + (_silu(h @ w["gate"].T) * (h @ w["up"].T)) @ w["down"].T
    return x


def _exact_transformer(case, seed):
    g, config = _generator(seed), _transformer_config(case)
    weights = _transformer_weights(case, g)
    head = _w4_f64(weights["lm_head"])
    logits = lambda x: _rms(x, weights["final_norm"], EPSILON) @ head.T
    embedded = lambda tokens: _f64(weights["embedding"][torch.as_tensor(np.asarray(tokens), device="cuda")])
    scale, kv, dim = case["head_dim"] ** -0.5, case["kv_heads"], case["head_dim"]
    if case["kind"] == "w4_batch":
        pool, lengths, starts, _, tokens = _batch_inputs(case, g, config)
        offsets = [region[:2] for region in config.kv_layout.regions]

        def attend(index, q, k, v):
            out = []
            for b in range(case["batch"]):
                start, length = int(starts[b]), int(lengths[b])
                past = pool[start:start + length]
                parts = []
                for offset, own in zip(offsets[index], (k, v)):
                    at = config.token_elements + offset // GROUP * 2
                    chosen = torch.cat([past[:, offset:offset + kv * dim], past[:, at:at + kv * dim // GROUP * 2]], dim=1)
                    parts.append(torch.cat([_unpacked(chosen, kv * dim).view(length, kv, dim), own[b:b + 1]]))
                out.append(_attend(q[b:b + 1], *parts, scale, torch.ones(1, length + 1, dtype=torch.bool, device="cuda")))
            return torch.cat(out)

        return {"logits": logits(_transformer_layers(case, weights, embedded(tokens.cpu().numpy()), lengths.cpu().numpy(), attend))}
    count = case["tokens"] if case["kind"] == "w4_prompt" else case["context"]
    tokens, cache, at = _tokens(case, seed, count + 1), [], _places(count)

    def attend_prompt(index, q, k, v):
        if case["kind"] == "w4_token":
            cache.append((_quantised(k), _quantised(v)))
        return _attend(q, k, v, scale, at[None, :] <= at[:, None])

    x = _transformer_layers(case, weights, embedded(tokens[:count]), np.arange(count), attend_prompt)
    if case["kind"] == "w4_prompt":
        return {"logits": logits(x[-1:])}
    seen = torch.ones(1, count + 1, dtype=torch.bool, device="cuda")
    attend_token = lambda index, q, k, v: _attend(q, torch.cat([cache[index][0], k]), torch.cat([cache[index][1], v]), scale, seen)
    x = _transformer_layers(case, weights, embedded(tokens[count:]), np.array([count]), attend_token)
    return {"logits": logits(x)[0]}


def _convolved(x, w, bias=0.0):
    """Per channel over time, the current token last."""
    taps = w.shape[1]
    padded = torch.cat([torch.zeros(taps - 1, x.shape[1], dtype=x.dtype, device=x.device), x])
    return sum(padded[i:i + x.shape[0]] * w[:, i] for i in range(taps)) + bias


def _recurrent_mixer(h, m, w, eps):
    t, heads, e, n = h.shape[0], m.heads, m.vdim, m.state
    p = h @ w("in").T
    z, mixed, dt = p[:, :m.inner], p[:, m.inner:m.inner + m.channels], p[:, m.inner + m.channels:]
    mixed = _silu(_convolved(mixed, w("conv"), w("conv.b")))
    x = mixed[:, :m.inner].view(t, heads, e)
    per = heads // m.groups
    b, c = (part.reshape(t, m.groups, n).repeat_interleave(per, dim=1) for part in mixed[:, m.inner:].chunk(2, dim=1))
    dt = torch.nn.functional.softplus(dt + w("dt_bias"))
    decay = torch.exp(-torch.exp(w("A_log")) * dt)
    state, y = torch.zeros(heads, n, e, dtype=h.dtype, device=h.device), torch.empty_like(x)
    for i in range(t):
        state = decay[i, :, None, None] * state + b[i, :, :, None] * (dt[i, :, None] * x[i])[:, None, :]
        y[i] = (c[i, :, None, :] @ state)[:, 0]
    y = (y + w("D")[:, None] * x).reshape(t, -1) * _silu(z)
    parts = y.view(t, m.norm_groups, -1)
    parts = parts / torch.sqrt(parts.square().mean(-1, keepdim=True) + eps)
    return (parts.reshape(t, -1) * w("norm")) @ w("o").T


def _gated(h, w, prefix, act):
    return (act(h @ w(prefix + "gate").T) * (h @ w(prefix + "up").T)) @ w(prefix + "down").T


def _routed(h, f, w):
    chosen = torch.topk(h @ w("router").T, f.top, dim=1)
    weights, out = torch.softmax(chosen.values, dim=1), torch.sigmoid(h @ w("shared.sg").T) * _gated(h, w, "shared.", _silu)
    for e in range(f.experts):
        rows, place = torch.nonzero(chosen.indices == e, as_tuple=True)
        out.index_add_(0, rows, weights[rows, place, None] * _gated(h[rows], w, f"e{e}.", _silu))
    return out


def _exact_barovik(parsed, get, x):
    t, first = x.shape[0], None
    at = _places(t)
    for index, layer in enumerate(parsed.layers):
        m, w = layer.mixer, lambda name: get(f"l{index}.mix.{name}")
        h = _rms(x, get(f"l{index}.norm1"), parsed.epsilon)
        if hasattr(m, "chunk"):
            q, k, v = ((h @ w(name).T).view(t, -1, m.dim) for name in "qkv")
            if first is None:
                first = v
            else:
                v = (1 - w("vmix")) * v + w("vmix") * first
            seen = (at[None, :] <= at[:, None]) & (at[None, :] // m.chunk == at[:, None] // m.chunk)
            x = x + _attend(q, k, v, m.scale, seen, m.softcap, w("sink")).reshape(t, -1) @ w("o").T
        else:
            x = x + _recurrent_mixer(h, m, w, parsed.epsilon)
        w = lambda name: get(f"l{index}.mlp.{name}")
        h = _rms(x, get(f"l{index}.norm2"), parsed.epsilon)
        x = x + (_routed(h, layer.ffn, w) if hasattr(layer.ffn, "experts") else
                 _gated(h, w, "", lambda z: torch.nn.functional.gelu(z, approximate="tanh")))
    return _rms(x[-1:], get("final.norm"), parsed.epsilon) @ get("head").T


def _turned(x, r):
    angle = _places(x.shape[0]).double()[:, None, None] * torch.from_numpy(r.frequencies).cuda()
    half, cos, sin = r.dims // 2, torch.cos(angle), torch.sin(angle)
    a, b = x[..., :half], x[..., half:r.dims]
    return torch.cat([a * cos - b * sin, b * cos + a * sin, x[..., r.dims:]], dim=-1)


def _window_mixer(h, m, w, eps):
    t, at = h.shape[0], _places(h.shape[0])
    q, k = (_turned(_rms((h @ w(name).T).view(t, -1, m.dim), w(name + ".norm"), eps), m.rotation) for name in "qk")
    back = at[:, None] - at[None, :]
    return _attend(q, k, (h @ w("v").T).view(t, -1, m.vdim), m.scale, (back >= 0) & (back < m.window)).reshape(t, -1) @ w("o").T


def _delta_mixer(h, m, w, eps):
    t, per = h.shape[0], m.heads // m.kv_heads
    q, k, v = (_silu(_convolved(h @ w(name).T, w(name + ".conv"))).view(t, -1, size) for name, size in zip("qkv", (m.dim, m.dim, m.vdim)))
    unit = lambda x: x / torch.sqrt(x.square().sum(-1, keepdim=True) + 1e-6)
    q, k = ((unit(x) * gain).repeat_interleave(per, dim=1) for x, gain in ((q, m.dim ** -0.5), (k, 1.0)))
    step = torch.nn.functional.softplus(h @ w("a1").T @ w("a2").T + w("dt_bias")).view(t, m.heads, m.dim)
    decay, beta = torch.exp(-torch.exp(w("A_log"))[None, :, None] * step), torch.sigmoid(h @ w("b").T)
    state, out = torch.zeros(m.heads, m.dim, m.vdim, dtype=h.dtype, device=h.device), torch.empty_like(v)
    for i in range(t):
        state = decay[i, :, :, None] * state
        u = beta[i, :, None] * (v[i] - (k[i, :, None, :] @ state)[:, 0])
        state = state + k[i, :, :, None] * u[:, None, :]
        out[i] = (q[i, :, None, :] @ state)[:, 0]
    gate = torch.sigmoid(h @ w("g1").T @ w("g2").T).view(t, m.heads, m.vdim)
    return (_rms(out, w("norm"), eps) * gate).reshape(t, -1) @ w("o").T


def _exact_koketar(parsed, get, x):
    eps, gain = parsed.epsilon, parsed.residual_scale
    for index, layer in enumerate(parsed.layers):
        m, p = layer.mixer, f"l{index}."
        y = m.left_scale * _window_mixer(x, m.left, lambda name: get(p + "mix.left." + name), eps) + \
            m.right_scale * _delta_mixer(x, m.right, lambda name: get(p + "mix.right." + name), eps)
        x = x + gain * _rms(y, 1 + get(p + "norm1"), eps)
        limit = layer.ffn.limit
        g = torch.clamp(x @ get(p + "mlp.gate").T, max=limit)
        u = torch.clamp(x @ get(p + "mlp.up").T, -limit, limit)
        y = (g * torch.sigmoid(1.702 * g) * (u + 1)) @ get(p + "mlp.down").T
        x = x + gain * _rms(y, 1 + get(p + "norm2"), eps)
    logits = _rms(x[-1:], 1 + get("final.norm"), eps) @ get("embed").T
    return parsed.logit_softcap * torch.tanh(logits / parsed.logit_softcap)


def _exact_layered(case, seed):
    parsed, tensors = _layered_weights(case, seed)
    get = lambda name: _f64(tensors[name])
    tokens = torch.from_numpy(_tokens(case, seed, case["tokens"] + case.get("reply", 0))).cuda()
    logits = (_exact_barovik if case["design"] == "Barovik" else _exact_koketar)(parsed, get, get("embed")[tokens])
    return {"logits": logits if case["kind"] == "layered_prompt" else logits[0]}


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        x, packed, scale, bias = _linear_inputs(case, seed)
        y = _f64(x) @ _w4_f64((packed, scale)).T
        return y if bias is None else y + _f64(bias)
    if kind == "cache_attention":
        return _exact_cache_attention(case, seed)
    if kind == "prompt_attention":
        return _exact_prompt_attention(case, seed)
    return _exact_transformer(case, seed) if kind.startswith("w4") else _exact_layered(case, seed)
