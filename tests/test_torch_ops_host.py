"""The torch operator's native side is an addition: the HIP library is built and the operator registered without it."""
import os
import subprocess
import sys
import types

import pytest

from llmopt_amd import build

torch = pytest.importorskip("torch")
ROOT = os.path.join(os.path.dirname(__file__), "..")


@pytest.mark.parametrize("missing", ["torch for ROCm", "ROCm's folder", "g++", "a header", "nothing"])
def test_the_hip_library_is_built_without_the_operator(monkeypatch, tmp_path, missing):
    from torch.utils import cpp_extension
    ran = []

    def run(command, **_):
        ran.append(command[0])
        if command[0] == "g++" and missing == "g++":
            raise FileNotFoundError("g++")
        if command[0] == "g++" and missing == "a header":
            return types.SimpleNamespace(returncode=1, stderr="no such header")
        (tmp_path / os.path.basename(command[command.index("-o") + 1])).touch()
        return types.SimpleNamespace(returncode=0, stderr="")

    (tmp_path / "a.o").touch()
    monkeypatch.setattr(build, "_compile", lambda *_: str(tmp_path / "a.o"))
    monkeypatch.setattr(build, "LIBRARY", str(tmp_path / "libllmopt_hip.so"))
    monkeypatch.setattr(build, "HERE", str(tmp_path))
    monkeypatch.setattr(build.subprocess, "run", run)
    if missing == "torch for ROCm":
        monkeypatch.setattr(torch.version, "hip", None)
    if missing == "ROCm's folder":
        monkeypatch.setattr(cpp_extension, "ROCM_HOME", None)
    stale = tmp_path / os.path.basename(build.torch_library(torch.__version__))
    stale.touch()
    assert build.build(force=True) == str(tmp_path / "libllmopt_hip.so")
    assert os.path.exists(tmp_path / "libllmopt_hip.so") and ran[-1] == "hipcc"
    assert ran[:-1] == ([] if missing in ("torch for ROCm", "ROCm's folder") else ["g++"])
    assert stale.exists() == (missing not in ("g++", "a header"))  # (none of an older source is left)


def test_the_operators_library_is_of_one_torch():
    assert build.torch_library("2.10.0+rocm7.0") != build.torch_library("2.10.1+rocm7.0")


def test_the_operator_without_its_native_side():
    code = """
import warnings
from llmopt_amd import build
build.torch_library = lambda version: "/nonexistent/libllmopt_torch.so"
with warnings.catch_warnings(record=True) as told:
    warnings.simplefilter("always")
    from llmopt_amd import torch_ops
import torch
assert torch_ops._native is None and any("longer way" in str(w.message) for w in told)
assert torch._C._dispatch_has_kernel_for_dispatch_key("llmopt::w4a16_linear", "CUDA")
meta = lambda *shape, dtype=torch.float16: torch.empty(shape, dtype=dtype, device="meta")
assert torch.ops.llmopt.w4a16_linear(meta(5, 64), meta(8, 32, dtype=torch.uint8), meta(8, 1), None).shape == (5, 8)
"""
    subprocess.run([sys.executable, "-c", code], cwd=ROOT, check=True, timeout=300)
