"""Which of its graphs a retained plan runs, without a GPU: plan.cpp over stand-ins for HIP (plan_host.cpp)."""
import ctypes
import os
import subprocess
import threading

import pytest

ROOT = os.path.join(os.path.dirname(__file__), "..")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    library = str(tmp_path_factory.mktemp("plan") / "plan.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-pthread", "-w", "-D__HIP_PLATFORM_AMD__", "-I", f"{ROCM}/include",
                    "-I", os.path.join(ROOT, "llmopt_amd", "csrc"), os.path.join(os.path.dirname(__file__), "plan_host.cpp"),
                    "-Wl,-Bsymbolic", "-o", library], check=True)
    loaded = ctypes.CDLL(library)
    for name, result, arguments in (("stub_plan", ctypes.c_void_p, [ctypes.c_char_p]),
                                    ("stub_step", ctypes.c_long, [ctypes.c_void_p, ctypes.c_long]),
                                    ("stub_recapture", None, [ctypes.c_void_p]),
                                    ("stub_next_tag", None, [ctypes.c_void_p, ctypes.c_uint32]),
                                    ("stub_launches", ctypes.c_long, [ctypes.c_void_p, ctypes.c_long]),
                                    ("llmopt_hip_prebaked_resident_layers", ctypes.c_int, [ctypes.c_void_p]),
                                    ("llmopt_hip_release_prebaked", None, [ctypes.c_void_p])):
        getattr(loaded, name).restype, getattr(loaded, name).argtypes = result, arguments
    return loaded


def tags(stub):
    out = (ctypes.c_uint32 * 4096)()
    return list(out[:stub.stub_launches(out, 4096)])


def test_plans_and_their_graphs(stub):
    for name, layers in ((b"layers", 4), (b"other", 0)):
        stub.stub_set(96, 4, 0, 0)
        plan = stub.stub_plan(name)
        assert stub.llmopt_hip_prebaked_resident_layers(plan) == layers
        assert [stub.stub_step(plan, token) for token in (5, 6, 7)] == [6, 7, 8]
        assert tags(stub) == ([1, 6, 11] if layers else [0, 0, 0])
        stub.llmopt_hip_release_prebaked(plan)
        assert stub.stub_live_graphs() == 0


def test_a_step_that_gives_up_and_all_behind_it_run_by_launches(stub):
    stub.stub_set(96, 4, 0, 1)
    plan = stub.stub_plan(b"layers")
    assert [stub.stub_step(plan, 5), stub.stub_step(plan, 6)] == [6, 7]
    assert tags(stub) == [1, 0, 0] and stub.llmopt_hip_prebaked_resident_layers(plan) == 0
    stub.llmopt_hip_release_prebaked(plan)


@pytest.mark.parametrize("when", ["created", "captured again"])
def test_a_plan_whose_second_graph_fails_keeps_its_launches(stub, when):
    stub.stub_set(96, 4, when == "created", 0)
    plan = stub.stub_plan(b"layers")
    assert plan is not None
    if when == "captured again":
        assert stub.stub_step(plan, 5) == 6 and tags(stub) == [1]
        stub.stub_set(96, 4, 1, 0)
        stub.stub_recapture(plan)
    assert [stub.stub_step(plan, 6), stub.stub_step(plan, 7)] == [7, 8]
    assert tags(stub) == [0, 0] and stub.llmopt_hip_prebaked_resident_layers(plan) == 0
    stub.llmopt_hip_release_prebaked(plan)
    assert stub.stub_live_graphs() == 0


def test_tags_come_round_over_cleared_words(stub):
    """A step's tags never meet words that carry them from before: they start over at 1 behind a clearing of all words."""
    stub.stub_set(96, 64, 0, 0)
    plan = stub.stub_plan(b"layers")
    near = 0xffffff00 - 65
    stub.stub_next_tag(plan, near - 65)
    cleared = []
    for token in range(5):
        stub.stub_step(plan, token)
        cleared.append(stub.stub_cleared())
    # (the clearing is queued in front of the last step of the old tags; that step's own are below 2^32)
    assert tags(stub) == [near - 65, near, near + 65, 1, 66] and near + 65 + 64 < 2 ** 32
    assert cleared == [0, 0, 1, 1, 1]
    stub.llmopt_hip_release_prebaked(plan)


@pytest.mark.parametrize("workgroups, most", [([96, 96], 192), ([96] * 5, 192), ([129, 128], 129), ([121, 128], 249), ([256] * 3, 256),
                                              ([96, 256, 24, 40, 96], 256)])
def test_resident_launches_of_several_threads(stub, workgroups, most):
    """Every step of every plan is resident, whatever other threads do; launches share the device as long as all their workgroups,
    in whole sets of eight, find room."""
    plans = []
    for count in workgroups:
        stub.stub_set(count, 4, 0, 0)
        plans.append(stub.stub_plan(b"layers"))
    stub.stub_set(0, 4, 0, 0)

    def steps(plan):
        for token in range(30):
            assert stub.stub_step(plan, token) == token + 1

    threads = [threading.Thread(target=steps, args=(plan,)) for plan in plans]
    for thread in threads:
        thread.start()
    for thread in threads:
        thread.join()
    assert sorted(tags(stub)) == sorted(1 + 5 * step for step in range(30) for _ in plans)
    assert max(workgroups) <= stub.stub_most_under_way() <= 256
    if len(set(workgroups)) <= 2:
        assert stub.stub_most_under_way() == most
    for plan in plans:
        stub.llmopt_hip_release_prebaked(plan)
