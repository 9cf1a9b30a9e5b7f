"""`torch.ops.llmopt.w4a16_linear` (python/llmopt_backend/quantization.py:174-185) on ROCm tensors."""
import numpy as np
import pytest

import oracle
from tests.gpu_util import assert_close_to_oracle, w4_case

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def op():
    import llmopt_amd.torch_ops  # noqa: F401  (registers the operator)
    return torch.ops.llmopt.w4a16_linear


@pytest.mark.parametrize("shape,n,k,bias", [((1, 576), 1536, 576, False), ((2, 3, 576), 192, 576, True),
                                            ((40, 1024), 1000, 1024, True)])
def test_matches_oracle(op, shape, n, k, bias):
    rng = np.random.default_rng(n)
    x, packed, scale, b = w4_case(rng, int(np.prod(shape[:-1])), n, k, bias=bias)
    device = torch.device("cuda:0")
    tx = torch.from_numpy(x.reshape(shape)).to(device)
    out = op(tx, torch.from_numpy(packed).to(device), torch.from_numpy(scale).to(device),
             torch.from_numpy(b).to(device) if bias else None)
    assert out.shape == (*shape[:-1], n) and out.dtype == torch.float16
    expected = oracle.w4a16_linear(x, packed, scale, b)
    assert_close_to_oracle(out.cpu().numpy().reshape(-1, n), expected, "torch op")


def test_reference_golden_fixture(op, golden):
    """python/tests/test_quantization.py:43-55 / python/examples/w4a16_linear_fx.json."""
    case = golden["w4a16_linear_fixture"]
    device = torch.device("cuda:0")
    packed = np.arange(96, dtype=np.uint8).reshape(3, 32)
    packed[0, 0] = 0x78
    scale = np.array(case["scale"], dtype=np.float16).reshape(3, 1)
    bias = np.array(case["bias"], dtype=np.float16)
    x = torch.ones((2, 64), dtype=torch.float16, device=device)
    out = op(x, torch.from_numpy(packed).to(device), torch.from_numpy(scale).to(device),
             torch.from_numpy(bias).to(device))
    assert out.cpu().numpy().view(np.uint16).reshape(-1).tolist() == case["expected_output_bits"]


def test_argument_checks(op):
    device = torch.device("cuda:0")
    packed = torch.zeros((8, 32), dtype=torch.uint8, device=device)
    scale = torch.ones((8, 1), dtype=torch.float16, device=device)
    with pytest.raises(TypeError, match="activations must be torch.float16"):
        op(torch.zeros((1, 64), dtype=torch.float32, device=device), packed, scale, None)
    with pytest.raises(TypeError, match="storage must be torch.uint8"):
        op(torch.zeros((1, 64), dtype=torch.float16, device=device), packed.to(torch.int8), scale, None)
    with pytest.raises(ValueError, match="scales must have shape"):
        op(torch.zeros((1, 64), dtype=torch.float16, device=device), packed, scale.reshape(1, 8), None)


def test_meta_kernel(op):
    out = op(torch.empty((5, 64), dtype=torch.float16, device="meta"),
             torch.empty((8, 32), dtype=torch.uint8, device="meta"),
             torch.empty((8, 1), dtype=torch.float16, device="meta"), None)
    assert out.shape == (5, 8) and out.dtype == torch.float16


def test_calls_in_a_row_on_one_and_on_alternating_streams(op):
    """Nothing waits between calls on one stream, not even where they share the context's scratch memory (8 rows of K =
    14336 and 130 of K = 16384 over few columns: K split over workgroups); a stream's calls come after those before."""
    rng = np.random.default_rng(3)
    device = torch.device("cuda:0")
    cases = [w4_case(rng, m, n, k, bias=True) for m, n, k in ((1, 576, 576), (8, 256, 14336), (130, 128, 16384), (24, 1000, 4096))]
    tensors = [[torch.from_numpy(a).to(device) for a in case] for case in cases]
    torch.cuda.synchronize()
    streams = [torch.cuda.current_stream(), torch.cuda.Stream(), torch.cuda.Stream()]
    outs = []
    for turn in range(24):
        with torch.cuda.stream(streams[turn // 8]):
            outs.append(op(*tensors[turn % 4]))
        if turn % 8 == 7 and turn // 8 + 1 < len(streams):
            streams[turn // 8 + 1].wait_stream(streams[turn // 8])
    for turn in range(6):
        with torch.cuda.stream(streams[turn % 3]):
            outs.append(op(*tensors[turn % 4]))
    torch.cuda.synchronize()
    for turn, out in enumerate(outs):
        case = (turn if turn < 24 else turn - 24) % 4
        assert_close_to_oracle(out.cpu().numpy(), oracle.w4a16_linear(*cases[case]), f"call {turn}")


def test_refused_shapes(op):
    device = torch.device("cuda:0")
    half = lambda *shape: torch.zeros(shape, dtype=torch.float16, device=device)
    with pytest.raises(RuntimeError):
        op(half(3, 0), torch.zeros((8, 0), dtype=torch.uint8, device=device), half(8, 0), None)
    with pytest.raises(RuntimeError):
        op(half(3, 64), torch.zeros((0, 32), dtype=torch.uint8, device=device), half(0, 1), None)
    assert op(half(0, 64), torch.zeros((8, 32), dtype=torch.uint8, device=device), half(8, 1), None).shape == (0, 8)


@pytest.mark.parametrize("same", [False, True])
def test_a_stream_under_capture_is_refused(op, same):
    """The first call on a stream that is being captured, after calls on it or on another one, is an error that leaves
    the capture whole: what else is recorded replays, and the operator goes on outside."""
    rng = np.random.default_rng(4)
    device = torch.device("cuda:0")
    case = w4_case(rng, 8, 256, 14336)  # K split over workgroups: the context's scratch memory is in use
    tensors = [torch.from_numpy(a).to(device) for a in case[:3]] + [None]
    x = torch.arange(100, dtype=torch.float32, device=device)
    torch.cuda.synchronize()
    warm, captured = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(captured if same else warm):
        op(*tensors)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=captured):
        with pytest.raises(RuntimeError, match="captured"):
            op(*tensors)
        y = x + 1
    for turn in range(3):
        x += turn
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, x + 1)
        assert_close_to_oracle(op(*tensors).cpu().numpy(), oracle.w4a16_linear(*case[:3], None), "after the capture")


@pytest.mark.parametrize("layout", ["plain", "strided input", "strided weights", "offset input", "bias of two dimensions", "vector"])
def test_native_calls_and_those_left_to_python(op, layout, monkeypatch):
    """Once a device has a runtime, calls that need nothing but the launch never reach Python; the others give the same."""
    from llmopt_amd import torch_ops
    from llmopt_amd.native import LlmoptError
    in_python, check = [], torch_ops._check_arguments
    monkeypatch.setattr(torch_ops, "_check_arguments", lambda *args: in_python.append(args) or check(*args))
    rng = np.random.default_rng(11)
    device = torch.device("cuda:0")
    case = w4_case(rng, 4, 96, 128, bias=True)
    x, packed, scale, bias = (torch.from_numpy(a).to(device) for a in case)
    op(x, packed, scale, bias)
    in_python.clear()
    if layout == "strided input":
        x = torch.cat([x, x], dim=1)[:, :128]
    elif layout == "strided weights":
        packed, scale = torch.cat([packed, packed], dim=1)[:, :64], scale.t().contiguous().t()
    elif layout == "offset input":
        x = torch.cat([x, x])[4:]
    elif layout == "bias of two dimensions":
        bias = bias.reshape(2, 48)
    elif layout == "vector":
        x = x[0]
    for _ in range(2):
        out = op(x, packed, scale, bias)
        assert out.shape == (*x.shape[:-1], 96) and out.is_contiguous()
        want = oracle.w4a16_linear(*case)
        assert_close_to_oracle(out.cpu().numpy().reshape(-1, 96), want[:1] if layout == "vector" else want, layout)
    assert len(in_python) == (2 if layout.startswith("strided") else 0)
    with pytest.raises(ValueError, match="features"):
        op(x[..., :64].contiguous(), packed, scale, bias)
    with pytest.raises(TypeError, match="bias must be"):
        op(x, packed, scale, bias.float())
    with pytest.raises(LlmoptError):
        op(x.new_zeros((3, 64)), packed.new_zeros((0, 32)), scale.new_zeros((0, 1)), None)
    assert len(in_python) == (5 if layout.startswith("strided") else 3)


def test_a_closed_runtime_is_not_launched_from(op):
    """After its runtime is closed the operator says so, natively and from Python, and a new one takes the calls again."""
    from llmopt_amd import torch_ops
    from llmopt_amd.native import LlmoptError
    rng = np.random.default_rng(12)
    device = torch.device("cuda:0")
    case = w4_case(rng, 2, 64, 128, bias=False)
    tensors = [torch.from_numpy(a).to(device) for a in case[:3]]
    index = torch.cuda.current_device()
    op(*tensors, None)
    torch.cuda.synchronize()
    torch_ops._runtimes[index].close()
    for _ in range(2):
        with pytest.raises(LlmoptError, match="finalized"):
            op(*tensors, None)
    del torch_ops._runtimes[index]
    for _ in range(2):
        assert_close_to_oracle(op(*tensors, None).cpu().numpy(), oracle.w4a16_linear(*case[:3], None), "reopened")
