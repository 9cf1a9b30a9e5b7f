"""What a decode step writes to its state buffers, with a runtime that keeps buffers in host memory."""
import numpy as np
import pytest

from llmopt_amd.decode_step import DecodeConfig, DecodeStep, rope_rows


class HostBuffer:
    def __init__(self, memory):
        self.memory, self.byte_length = memory, len(memory)

    def view(self, offset, length):
        assert length > 0 and offset + length <= self.byte_length
        return HostBuffer(self.memory[offset:offset + length])

    def write(self, data, offset=0):
        data = np.ascontiguousarray(data).reshape(-1).view(np.uint8)
        self.memory[offset:offset + data.size] = data

    def numpy(self, dtype):
        return self.memory.copy().view(dtype)


class HostRuntime:
    def create_buffer(self, size):
        return HostBuffer(np.zeros(size, dtype=np.uint8))

    def buffer_of_bytes(self, data):
        buffer = self.create_buffer(np.asarray(data).nbytes)
        buffer.write(data)
        return buffer


CONFIG = DecodeConfig(hidden=64, q_heads=1, kv_heads=1, head_dim=64, mlp=64, layers=0, vocabulary=64, epsilon=1e-5)
LENGTHS, SLOTS, POSITIONS = np.array([5, 9, 300], dtype=np.uint32), np.array([7, 1, 4], dtype=np.uint32), np.array([6, 10, 301])


def step(lengths, slots, positions):
    runtime = HostRuntime()
    none = runtime.create_buffer(64)
    weights = dict(embedding=none, final_norm=none, lm_head=(none, none), layers=[])
    return DecodeStep(runtime, CONFIG, {}, 3, none, none, np.zeros(3, dtype=np.uint32), lengths, slots, positions,
                      max_context=1000, slots_host=np.arange(1000), device_weights=weights)


def every_other(a):
    return np.repeat(a, 2)[::2]


@pytest.mark.parametrize("form", [
    lambda a: a, list, every_other, lambda a: a[::-1].copy()[::-1], lambda a: a.reshape(3, 1), lambda a: a.astype(np.int64),
    lambda a: np.concatenate([a, a]),  # more entries than sequences: the others are not read
], ids=["array", "list", "every other", "reversed", "column", "int64", "longer"])
@pytest.mark.parametrize("which", [0, 1, 2, None])
def test_state_of_every_form_of_arrays(form, which):
    given = [form(a) if which in (index, None) else a for index, a in enumerate((LENGTHS, SLOTS, POSITIONS))]
    made = step(*given)
    np.testing.assert_array_equal(made.past_lengths.numpy(np.uint32)[:3], LENGTHS)
    np.testing.assert_array_equal(made.new_slots.numpy(np.uint32)[:3], SLOTS)
    for rows, expected in zip((made.cos, made.sin), rope_rows(CONFIG, POSITIONS)):
        np.testing.assert_array_equal(rows.numpy(np.float16)[:expected.size], expected.reshape(-1))


def test_state_after_steps():
    made = step(LENGTHS, SLOTS, POSITIONS)
    made.advance()
    made.seek(every_other(LENGTHS + 2), every_other(POSITIONS + 5))
    np.testing.assert_array_equal(made.past_lengths.numpy(np.uint32), LENGTHS + 2)
    np.testing.assert_array_equal(made.new_slots.numpy(np.uint32), LENGTHS + 2)
    for rows, expected in zip((made.cos, made.sin), rope_rows(CONFIG, POSITIONS + 5)):
        np.testing.assert_array_equal(rows.numpy(np.float16), expected.reshape(-1))
