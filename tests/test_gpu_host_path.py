"""What a decoded token's host side reads: halves widened on the host, the output word of a plan."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

@pytest.fixture(scope="module")
def runtime():
    from llmopt_amd.native import Runtime
    rt = Runtime()
    yield rt
    rt.close()


@pytest.mark.parametrize("count", [1, 7, 8, 9, 1023, 65536])
def test_widened_halves_are_the_halves(runtime, count):
    halves = np.arange(65536, dtype=np.uint32).astype(np.uint16)[-count:].view(np.float16)  # (65536: every half there is)
    out = runtime.buffer_of_bytes(halves).widened()
    with np.errstate(invalid="ignore"):
        expected = halves.astype(np.float32)
    number = ~np.isnan(expected)
    np.testing.assert_array_equal(np.isnan(out), ~number)
    np.testing.assert_array_equal(out[number].view(np.uint32), expected[number].view(np.uint32))


def test_widening_refuses_a_half_value(runtime):
    with pytest.raises(ValueError):
        runtime.buffer_of_bytes(np.zeros(3, dtype=np.uint8)).widened()


@pytest.mark.parametrize("wrapped", [False, True])  # (a wrapped pointer is read by a copy, memory of the context by a kernel)
def test_plan_hands_out_its_word(runtime, wrapped):
    from llmopt_amd.native import Prebaked
    from tests.gpu_util import u32s
    rows = runtime.create_buffer(4 * 300)
    logits = np.zeros(300, dtype=np.float32)
    token, out = runtime.create_buffer(8), runtime.create_buffer(4)
    output = runtime.wrap(out.device_pointer, 4) if wrapped else out
    plan = Prebaked(runtime, [("llmopt_argmax_f32", [rows, output], u32s(1, 300), (256, 1, 1), (256, 1, 1))], token, output)
    for best in (299, 0, 17):
        logits[:] = 0
        logits[best] = 1
        rows.write(logits)
        assert plan.execute(5, 0) == best


# each replay takes its own values, with and without a word to hand out, and beside steps of a second plan
@pytest.mark.parametrize("output", ["own", "wrapped", "short"])
def test_plan_takes_each_steps_token(runtime, output):
    from llmopt_amd.native import Prebaked
    from tests.gpu_util import u32s
    rows, best = runtime.buffer_of_bytes(np.arange(300, dtype=np.float32)), runtime.create_buffer(4)
    word = {"own": best, "wrapped": runtime.wrap(best.device_pointer, 4), "short": runtime.create_buffer(2)}[output]
    tokens = [runtime.create_buffer(8) for _ in range(2)]
    plans = [Prebaked(runtime, [("llmopt_argmax_f32", [rows, best], u32s(1, 300), (256, 1, 1), (256, 1, 1))], token, word)
             for token in tokens]
    for step in range(6):
        for number, plan in enumerate(plans):
            assert plan.execute(100 * number + step, 0) == (0 if output == "short" else 299)
            assert tokens[number].numpy(np.int64)[0] == 100 * number + step
