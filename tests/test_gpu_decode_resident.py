"""All layers of a decode step in one resident launch (a retained plan's, kernels/decode_resident.hip): several tokens
against the oracle chain and against the same records launched one by one."""
import numpy as np
import pytest

from oracle.chain import decode_chain
from tests.test_gpu_glue import pointwise_params
from tests.test_gpu_prebaked import build_step, make_case

pytestmark = pytest.mark.gpu

# sequences, their contexts, hidden, query and KV heads, mlp, layers
CASES = [
    ([2048], 576, 9, 3, 1536, 4),                                # one sequence, many runs
    ([0], 64, 1, 1, 64, 4),                                      # no context, the smallest sizes
    ([5, 64, 300], 576, 9, 3, 1536, 5),                          # launches of small batches
    ([15, 16, 17, 31, 33, 1, 0, 129, 700, 2, 64, 3, 8, 9, 10, 11], 320, 4, 2, 192, 4),  # a whole tile of sequences
    ([40 * i for i in range(17)], 576, 9, 3, 1536, 4),           # a sequence beyond a tile; five launches a layer
    ([3000] + [7 * i % 90 for i in range(47)], 256, 16, 4, 2048, 4),  # three tiles, one long context, the most heads
    ([9000], 64, 1, 1, 64, 4),                                   # more tokens a run than it holds slots of
    ([100, 90], 1024, 16, 1, 640, 4),                            # the widest rows, all heads on one KV head
]


@pytest.fixture(scope="module")
def runtime():
    from llmopt_amd.native import Runtime
    rt = Runtime()
    yield rt
    rt.close()


@pytest.mark.parametrize("lengths, hidden, q_heads, kv_heads, mlp, layers", CASES)
def test_resident_layers(runtime, lengths, hidden, q_heads, kv_heads, mlp, layers):
    from llmopt_amd.decode_step import DecodeConfig, random_weights
    from llmopt_amd.native import Prebaked
    print(f"resident layers m={len(lengths)} hidden={hidden} heads={q_heads}/{kv_heads} mlp={mlp} seed=3", flush=True)
    rng = np.random.default_rng(3)
    config = DecodeConfig(hidden=hidden, q_heads=q_heads, kv_heads=kv_heads, head_dim=64, mlp=mlp, layers=layers, vocabulary=500)
    weights = random_weights(config, rng)
    room, batch = 66, len(lengths)  # (launches take another form where no context can reach 64 tokens)
    case = make_case(rng, config, lengths, room)
    pool_host, slots, offsets, _, capacity, _ = case
    eager, eager_pool = build_step(runtime, config, weights, case, lengths, room)
    frozen, frozen_pool = build_step(runtime, config, weights, case, lengths, room)
    plan = Prebaked(runtime, frozen.dispatches, frozen.tokens, frozen.token_ids)
    assert plan.resident_layers == layers
    stride, elements = config.token_stride, config.token_elements
    tokens = rng.integers(0, config.vocabulary, batch)
    for index in range(3):
        past = np.asarray(lengths) + index
        new_slots = slots[offsets + past]
        eager.run(tokens)
        frozen.tokens.write(np.asarray(tokens, dtype=np.int64))
        before = frozen_pool.numpy(np.uint8).reshape(capacity, stride)
        first = plan.execute(int(tokens[0]), int(past[0]))
        got = frozen.work["x"][0].numpy(np.float16, (batch, hidden))
        assert first == int(frozen.token_ids.numpy(np.uint32)[0])
        want, _, want_pool = decode_chain(config, weights, before.reshape(-1).copy(), slots, offsets, past, new_slots, past, tokens)
        # Held to the oracle as the chain's launches are (4e-3), or, where a row's activations amplify every rounding in front of
        # them, to twice what the launches, rounded at the same places, are off there.
        other = eager.work["x"][0].numpy(np.float16, (batch, hidden)).astype(np.float64)
        want, got = np.asarray(want, dtype=np.float64), got.astype(np.float64)
        norm, rms = np.linalg.norm(want), np.sqrt(np.mean(want ** 2))
        assert np.isfinite(got).all() and np.linalg.norm(got - want) <= 4e-3 * norm
        assert np.abs(got - want).max() <= max(2e-2 * rms, 2 * np.abs(other - want).max())
        after = frozen_pool.numpy(np.uint8).reshape(capacity, stride)
        untouched = np.ones(capacity, dtype=bool)
        untouched[new_slots] = False
        np.testing.assert_array_equal(after[untouched], before[untouched])
        # The first layer's keys and values come from the same rows: one quantum where a value lies between two.  Behind it a row
        # may be off by 2e-2 of its RMS, and so its keys and values; a group of 64 has a value of 2 RMS
        # or more, which its scale makes 127 quanta: 127 * 2e-2 / 2 = 1.3 for the value, as much for the scale, and the one.
        quanta = lambda rows: rows[new_slots, :elements].view(np.int8).astype(np.int32)
        off = np.abs(quanta(after) - quanta(want_pool.reshape(capacity, stride)))
        assert off[:, :2 * kv_heads * 64].max() <= 1 and off.max() <= 3
        frozen_pool.copy_to(eager_pool)  # one quantum's difference must not grow into another continuation
        tokens = rng.integers(0, config.vocabulary, batch)
        eager.advance()
        frozen.advance()
    assert plan.resident_layers == layers  # no launch gave up


@pytest.mark.parametrize("lengths", [[300], [20 * i for i in range(11)]])
def test_thirty_layers(runtime, lengths):
    """The depth of a real model, held to the oracle as the chain's launches are."""
    from llmopt_amd.decode_step import DecodeConfig, random_weights
    from llmopt_amd.native import Prebaked
    rng = np.random.default_rng(8)
    config = DecodeConfig(hidden=256, q_heads=4, kv_heads=2, mlp=512, layers=30, vocabulary=500)
    weights = random_weights(config, rng)
    case = make_case(rng, config, lengths, 66)
    pool_host, slots, offsets, new_slots, capacity, batch = case
    eager, _ = build_step(runtime, config, weights, case, lengths, 66)
    frozen, frozen_pool = build_step(runtime, config, weights, case, lengths, 66)
    plan = Prebaked(runtime, frozen.dispatches, frozen.tokens, frozen.token_ids)
    assert plan.resident_layers == 30
    tokens = rng.integers(0, config.vocabulary, batch)
    eager.run(tokens)
    frozen.tokens.write(np.asarray(tokens, dtype=np.int64))
    plan.execute(int(tokens[0]), lengths[0])
    want, logits, _ = decode_chain(config, weights, pool_host.copy(), slots, offsets, lengths, new_slots, lengths, tokens)
    want = np.asarray(want, dtype=np.float64)
    got, launched = (step.work["x"][0].numpy(np.float16, want.shape).astype(np.float64) for step in (frozen, eager))
    off, launched_off = (np.linalg.norm(rows - want) / np.linalg.norm(want) for rows in (got, launched))
    print(f"30 layers: {off:.2e} off the oracle, the launches {launched_off:.2e}", flush=True)
    assert off <= 4e-3
    top, rms = frozen.token_ids.numpy(np.uint32, (batch,)), np.sqrt(np.mean(logits.astype(np.float64) ** 2))
    assert (logits[np.arange(batch), top] >= logits.max(axis=1) - 2e-2 * rms).all()
    after = frozen_pool.numpy(np.uint8).reshape(capacity, -1)
    untouched = np.setdiff1d(np.arange(capacity), new_slots)
    np.testing.assert_array_equal(after[untouched], pool_host.reshape(capacity, -1)[untouched])
    assert plan.resident_layers == 30


# what a workgroup's memory holds: 48 sequences of the widest rows, the most layers, and heads whose runs just fit beside them
@pytest.mark.parametrize("kv_heads, layers, resident", [(4, 64, 64), (2, 64, 0), (4, 65, 0)])
def test_most_memory(runtime, kv_heads, layers, resident):
    from llmopt_amd.decode_step import DecodeConfig, random_weights
    from llmopt_amd.native import Prebaked
    rng = np.random.default_rng(9)
    one = DecodeConfig(hidden=1024, q_heads=16, kv_heads=kv_heads, mlp=2048, layers=1, vocabulary=64)
    config = DecodeConfig(hidden=1024, q_heads=16, kv_heads=kv_heads, mlp=2048, layers=layers, vocabulary=64)
    weights = random_weights(one, rng)
    lengths = [3 * i for i in range(48)]
    case = make_case(rng, config, lengths, 66)
    first, _ = build_step(runtime, one, weights, case, lengths, 66)
    device = {**first.device, "layers": first.device["layers"] * layers}  # (one layer's weights for all)
    frozen, frozen_pool = build_step(runtime, config, {}, case, lengths, 66, device_weights=device)
    plan = Prebaked(runtime, frozen.dispatches, frozen.tokens, frozen.token_ids)
    assert plan.resident_layers == resident
    if resident == 0:
        return
    eager, eager_pool = build_step(runtime, config, {}, case, lengths, 66, device_weights=device)
    tokens = rng.integers(0, config.vocabulary, 48)
    eager.run(tokens)
    frozen.tokens.write(np.asarray(tokens, dtype=np.int64))
    plan.execute(int(tokens[0]), lengths[0])
    got, want = (step.work["x"][0].numpy(np.float16, (48, 1024)).astype(np.float64) for step in (frozen, eager))
    # two chains that round at the same places, each within the chain's tolerance
    assert np.isfinite(want).all() and np.linalg.norm(got - want) <= 8e-3 * np.linalg.norm(want)
    stride = config.token_stride
    untouched = np.setdiff1d(np.arange(case[4]), case[3])
    np.testing.assert_array_equal(frozen_pool.numpy(np.uint8).reshape(-1, stride)[untouched], case[0].reshape(-1, stride)[untouched])
    assert plan.resident_layers == 64


def small_plan(runtime, lengths, layers=5):
    from llmopt_amd.decode_step import DecodeConfig, random_weights
    from llmopt_amd.native import Prebaked
    rng = np.random.default_rng(11)
    config = DecodeConfig(hidden=192, q_heads=3, kv_heads=1, head_dim=64, mlp=256, layers=layers, vocabulary=300)
    weights = random_weights(config, rng)
    case = make_case(rng, config, lengths, 70)
    eager, eager_pool = build_step(runtime, config, weights, case, lengths, 70)
    frozen, frozen_pool = build_step(runtime, config, weights, case, lengths, 70)
    return eager, eager_pool, frozen, frozen_pool, Prebaked(runtime, frozen.dispatches, frozen.tokens, frozen.token_ids)


def step_pair(eager, frozen, plan, tokens):
    want = eager.run(tokens)
    frozen.tokens.write(np.asarray(tokens, dtype=np.int64))
    first = plan.execute(int(tokens[0]), int(frozen.host_lengths[0]))
    got = frozen.token_ids.numpy(np.uint32, (len(tokens),))
    assert first == int(got[0])
    eager.advance()
    frozen.advance()
    return want, got


@pytest.mark.parametrize("lengths", [[70], [70, 65, 3]])
def test_step_that_gives_up_is_run_by_launches(runtime, lengths, monkeypatch):
    """No wave waits for anything: the resident launch gives up, the step runs again launch by launch, bit for bit the
    eager one, and so do all behind it."""
    monkeypatch.setenv("LLMOPT_RESIDENT_WAIT_US", "0")
    eager, eager_pool, frozen, frozen_pool, plan = small_plan(runtime, lengths)
    assert plan.resident_layers == 5
    for _ in range(3):
        want, got = step_pair(eager, frozen, plan, [7] * len(lengths))
        assert plan.resident_layers == 0
        np.testing.assert_array_equal(got, want)
        np.testing.assert_array_equal(frozen.work["x"][0].numpy(np.uint16), eager.work["x"][0].numpy(np.uint16))
        np.testing.assert_array_equal(frozen_pool.numpy(np.uint8), eager_pool.numpy(np.uint8))


def test_only_scratch_between_the_records_is_left_out(runtime):
    """A buffer between the records that somebody may read: the plan launches every record and writes it."""
    from llmopt_amd.native import Prebaked
    eager, _, frozen, _, plan = small_plan(runtime, [70])
    assert plan.resident_layers == 5
    own = runtime.create_buffer(frozen.work["q_rot"].numpy(np.uint16).nbytes)
    dispatches = [(name, [own if b is frozen.work["q_rot"] else b for b in buffers], *rest)
                  for name, buffers, *rest in frozen.dispatches]
    plan = Prebaked(runtime, dispatches, frozen.tokens, frozen.token_ids)
    assert plan.resident_layers == 0
    step_pair(eager, frozen, plan, [7])
    np.testing.assert_array_equal(own.numpy(np.uint16), eager.work["q_rot"].numpy(np.uint16))
    # a record behind the layers that reads what one of them leaves
    x, stream = frozen.work["x"][0], frozen.work["stream"]
    last = (frozen.dispatches[-1][0], [stream, *frozen.dispatches[-1][1][1:]], *frozen.dispatches[-1][2:])
    assert Prebaked(runtime, [*frozen.dispatches[:-1], last], frozen.tokens, frozen.token_ids).resident_layers == 0


def test_plans_on_two_threads(runtime):
    """What a plan leaves does not depend on other threads: two plans stepped together leave, bit for bit, what each leaves alone,
    and no step runs by launches.  (One of several sequences takes the whole device, the other has to wait for it.)"""
    import threading
    from llmopt_amd.native import Runtime
    other = Runtime()
    try:
        for contexts in ([[70], [90]], [[70], [65, 90, 3]]):
            def steps(index, rt):
                _, _, frozen, pool, plan = small_plan(rt, contexts[index])
                left = []
                for token in range(40):
                    tokens = [token % 300] * len(contexts[index])
                    frozen.tokens.write(np.asarray(tokens, dtype=np.int64))
                    plan.execute(tokens[0], int(frozen.host_lengths[0]))
                    left.append(frozen.work["x"][0].numpy(np.uint16))
                    frozen.advance()
                assert plan.resident_layers == 5
                return np.stack(left), pool.numpy(np.uint8)

            alone = [steps(index, rt) for index, rt in enumerate((runtime, other))]
            together, failures = [None, None], []

            def on_a_thread(index, rt):
                try:
                    together[index] = steps(index, rt)
                except Exception as error:
                    failures.append(error)
            threads = [threading.Thread(target=on_a_thread, args=pair) for pair in enumerate((runtime, other))]
            for thread in threads:
                thread.start()
            for thread in threads:
                thread.join()
            assert not failures, failures
            for (x, pool), (same_x, same_pool) in zip(alone, together):
                np.testing.assert_array_equal(x, same_x)
                np.testing.assert_array_equal(pool, same_pool)
    finally:
        other.close()


def run_list(runtime, dispatches):
    batch = runtime.begin_batch()
    for name, buffers, parameters, grid, group in dispatches:
        batch.dispatch(name, buffers, parameters, grid=grid, group=group)
    batch.commit()


@pytest.mark.parametrize("lengths", [[70], [70, 65, 3]])
def test_layers_alone_that_give_up(runtime, lengths, monkeypatch):
    """Layers over rows that the host wrote, which are also the rows that come out: nothing in the plan writes them anew, so they
    must still be there for the launches."""
    from llmopt_amd.native import Prebaked
    monkeypatch.setenv("LLMOPT_RESIDENT_WAIT_US", "0")
    eager, eager_pool, frozen, frozen_pool, _ = small_plan(runtime, lengths)
    layers = frozen.dispatches[1:]
    plan = Prebaked(runtime, layers, frozen.tokens, frozen.token_ids)
    rows = np.random.default_rng(5).standard_normal((len(lengths), 192)).astype(np.float16)
    for _ in range(2):
        for step in (eager, frozen):
            step.work["x"][0].write(rows)
        run_list(runtime, eager.dispatches[1:])
        plan.execute(0, int(frozen.host_lengths[0]))
        np.testing.assert_array_equal(frozen.work["x"][0].numpy(np.uint16), eager.work["x"][0].numpy(np.uint16))
        np.testing.assert_array_equal(frozen.token_ids.numpy(np.uint32), eager.token_ids.numpy(np.uint32))
        np.testing.assert_array_equal(frozen_pool.numpy(np.uint8), eager_pool.numpy(np.uint8))


@pytest.mark.parametrize("place", ["in front", "behind", "both"])
def test_records_beside_the_layers_run_once(runtime, place, monkeypatch):
    """A record that reads what the step changes (an in-place add; a row that a later record replaces) must not run twice when the
    layers give up."""
    from llmopt_amd.native import Prebaked
    monkeypatch.setenv("LLMOPT_RESIDENT_WAIT_US", "0")
    eager, _, frozen, _, _ = small_plan(runtime, [70])
    h = eager.config.hidden
    params = pointwise_params((h,), (h,), (h,))
    one = np.full(h, 1.0, dtype=np.float16)

    def around(step):
        one_row, sum_row, other = (runtime.buffer_of_bytes(v) for v in (one, one * 2, one * 4))
        add = lambda left, right, out: ("llmopt_add_f16", [left, right, out], params, (h, 1, 1), (256, 1, 1))
        if place == "in front":
            return sum_row, [add(sum_row, one_row, sum_row), *step.dispatches]
        if place == "behind":
            return sum_row, [*step.dispatches, add(sum_row, one_row, sum_row)]
        # in front: other = sum + 1; behind: sum = other + 1
        return sum_row, [add(sum_row, one_row, other), *step.dispatches, add(other, one_row, sum_row)]

    want, eager_list = around(eager)
    got, frozen_list = around(frozen)
    plan = Prebaked(runtime, frozen_list, frozen.tokens, frozen.token_ids)
    eager.tokens.write(np.asarray([7], dtype=np.int64))
    for _ in range(2):
        run_list(runtime, eager_list)
        plan.execute(7, int(frozen.host_lengths[0]))
        np.testing.assert_array_equal(got.numpy(np.float16), want.numpy(np.float16))
        np.testing.assert_array_equal(frozen.work["x"][0].numpy(np.uint16), eager.work["x"][0].numpy(np.uint16))


def test_which_records_beside_the_layers_may_run_again(runtime):
    """The layers stay resident beside records that find what they read as it was (an add into the stream in front of the layers,
    behind the embedding that writes it anew), and not beside others."""
    from llmopt_amd.native import Prebaked
    _, _, frozen, _, _ = small_plan(runtime, [70])
    h, x = frozen.config.hidden, frozen.work["x"][0]
    params = pointwise_params((h,), (h,), (h,))
    row, out = (runtime.buffer_of_bytes(np.ones(h, dtype=np.float16)) for _ in range(2))
    add = lambda left, right, to: ("llmopt_add_f16", [left, right, to], params, (h, 1, 1), (256, 1, 1))
    resident = lambda records: Prebaked(runtime, records, frozen.tokens, frozen.token_ids).resident_layers
    embedding, *rest = frozen.dispatches
    assert resident([embedding, add(x, row, x), *rest]) == 5
    assert resident([embedding, *rest, add(row, row, out)]) == 5
    assert resident([embedding, *rest, add(row, row, row)]) == 0
    assert resident(rest) == 0                               # rows from outside, which the result replaces
    assert resident([embedding, *rest, add(row, row, x)]) == 5
    half = x.view(0, h)                                      # half of the rows written anew
    assert resident([("llmopt_add_f16", [row, row, half], pointwise_params((h // 2,), (h // 2,), (h // 2,)),
                      (h, 1, 1), (256, 1, 1)), *rest]) == 0
    # rows written into a buffer of their own: the result replaces nothing that is read
    own = runtime.create_buffer(h * 2)
    first = (rest[0][0], [own, *rest[0][1][1:]], *rest[0][2:])
    assert resident([first, *rest[1:]]) == 5


# slot table offsets, contexts, and the slot table's entry that the new token takes; the sizes of the layers
@pytest.mark.parametrize("offsets, lengths, new, shape", [
    ([0, 0, 0], [70, 71, 72], [70, 71, 72], (192, 3, 1, 256)),   # consecutive tokens of one sequence
    ([0, 100], [70, 90], [70, 5], (192, 3, 1, 256)),             # one sequence's new token in another's context
    ([0], [70], [69], (192, 3, 1, 256)),                         # in its own, the last token
    ([0], [9000], [1200], (64, 1, 1, 64)),                       # behind those slots of a run that the launch keeps at hand
])
def test_slots_that_the_step_itself_writes(runtime, offsets, lengths, new, shape):
    """The new tokens are in the cache before any sequence reads it: such a step runs by launches."""
    from llmopt_amd.decode_step import DecodeConfig, random_weights
    from llmopt_amd.native import Prebaked
    rng = np.random.default_rng(23)
    hidden, q_heads, kv_heads, mlp = shape
    config = DecodeConfig(hidden=hidden, q_heads=q_heads, kv_heads=kv_heads, head_dim=64, mlp=mlp, layers=4, vocabulary=300)
    weights = random_weights(config, rng)
    pool, slots, *_, capacity, _ = make_case(rng, config, [offsets[-1] + lengths[-1]], 70)
    case = pool, slots, np.asarray(offsets, np.uint32), slots[np.asarray(new)], capacity, len(lengths)
    eager, eager_pool = build_step(runtime, config, weights, case, lengths, 70)
    frozen, frozen_pool = build_step(runtime, config, weights, case, lengths, 70)
    plan = Prebaked(runtime, frozen.dispatches, frozen.tokens, frozen.token_ids)
    assert plan.resident_layers == 4
    tokens = rng.integers(0, config.vocabulary, len(lengths))
    for _ in range(2):
        want = eager.run(tokens)
        frozen.tokens.write(np.asarray(tokens, dtype=np.int64))
        assert plan.execute(int(tokens[0]), lengths[0]) == int(want[0])
        assert plan.resident_layers == 0
        np.testing.assert_array_equal(frozen.work["x"][0].numpy(np.uint16), eager.work["x"][0].numpy(np.uint16))
        np.testing.assert_array_equal(frozen_pool.numpy(np.uint8), eager_pool.numpy(np.uint8))
