"""`torch.ops.llmopt.w4a16_linear` on MI355X.

The reference registers
`w4a16_linear(Tensor input, Tensor packed_weight, Tensor scale, Tensor? bias) -> Tensor`
in the `llmopt` namespace (python/llmopt_backend/quantization.py:174-185) and
backs it with its native runtime (native/metal_runtime.cpp:139-147).  This
module registers the same schema for ROCm tensors: the kernel runs on the
tensors' own device memory (no copies), is queued on torch's current stream
and nothing waits for it.  Calls with nothing to refuse or lay out anew are native
code from torch's dispatcher on (csrc/torch/linear_op.cpp); the others come here, and all of
them where that code is not built for the installed torch.

    import llmopt_amd.torch_ops            # registers the operator
    y = torch.ops.llmopt.w4a16_linear(x, packed, scale, bias)

Same argument checks as the reference (quantization.py:104-118,144-147): fp16
activations and bias, uint8 `[N, K/2]` weights, fp16 `[N, K/64]` scales.
"""
from __future__ import annotations

import ctypes
import functools
import struct
import threading
import warnings
from typing import Optional

import torch

from .build import torch_library
from .native import Runtime, lib

GROUP_SIZE = 64
_ONE_ROW, _ROWS = b"llmopt_w4a16_linear_f16_g64", b"llmopt_w4a16_linear_f16_g64_m4"
_PARAMETERS = struct.Struct("<5I").pack  # m, n, k, has_bias, bias_row_stride
_library: Optional[torch.library.Library] = None
_native: Optional[ctypes.CDLL] = None
_runtimes: dict[int, Runtime] = {}
_lock = threading.Lock()


class _OperatorRuntime(Runtime):
    """A device's runtime: the native side launches from it until it is closed, and calls behind that say that it is."""

    def __init__(self, device: int):
        super().__init__(device=device)
        if _native is None:
            return
        self._unbind = functools.partial(_native.llmopt_torch_bind, device, None, None)
        # further calls on this device that need nothing but the launch no longer come here
        _native.llmopt_torch_bind(device, self.library, ctypes.cast(lib().llmopt_hip_launch, ctypes.c_void_p))

    def close(self) -> None:
        unbind = self.__dict__.pop("_unbind", None)
        if unbind is not None:
            unbind()
        super().close()


def _runtime(device_index: int) -> Runtime:
    runtime = _runtimes.get(device_index)
    if runtime is not None:
        return runtime
    with _lock:
        runtime = _runtimes.get(device_index)
        if runtime is None:
            runtime = _OperatorRuntime(device_index)
            _runtimes[device_index] = runtime
        return runtime


def _check_arguments(input, packed_weight, scale, bias):
    if packed_weight.dim() != 2:
        raise ValueError(f"packed W4 weight must be 2-D, got shape {tuple(packed_weight.shape)}")
    output_features, packed_k = packed_weight.shape
    logical_k = packed_k * 2
    if logical_k % GROUP_SIZE != 0:
        raise ValueError(f"W4 K dimension {logical_k} is not a multiple of the group size {GROUP_SIZE}")
    groups = logical_k // GROUP_SIZE
    if packed_weight.dtype != torch.uint8:
        raise TypeError(f"packed W4 weight storage must be torch.uint8, got {packed_weight.dtype}")
    if scale.dtype != torch.float16:
        raise TypeError(f"W4 scales must be torch.float16, got {scale.dtype}")
    if tuple(scale.shape) != (output_features, groups):
        raise ValueError(f"W4 scales must have shape [{output_features}, {groups}], got {tuple(scale.shape)}")
    if input.dtype != torch.float16:
        raise TypeError(f"W4A16 activations must be torch.float16, got {input.dtype}")
    if bias is not None and bias.dtype != torch.float16:
        raise TypeError(f"W4A16 bias must be torch.float16, got {bias.dtype}")
    if input.shape[-1] != logical_k:
        raise ValueError(f"W4A16 input has {input.shape[-1]} features, the weight expects {logical_k}")
    if bias is not None and bias.numel() != output_features:
        raise ValueError(f"W4A16 bias must have {output_features} elements, got {bias.numel()}")
    return output_features, logical_k


def _w4a16_linear_hip(input, packed_weight, scale, bias=None):
    n, k = _check_arguments(input, packed_weight, scale, bias)
    x, packed_weight, scale = input.contiguous(), packed_weight.contiguous(), scale.contiguous()
    m = x.numel() // k if k else x.view(-1, k).shape[0]
    output = torch.empty((*input.shape[:-1], n), dtype=torch.float16, device=input.device)
    if m == 0:
        return output
    addend = bias.contiguous() if bias is not None else scale
    runtime = _runtime(input.device.index if input.device.index is not None else torch.cuda.current_device())
    # queued on torch's stream; the tensors above outlive the launch call
    runtime.launch(_ONE_ROW if m == 1 else _ROWS,
                   (x.data_ptr(), packed_weight.data_ptr(), scale.data_ptr(), addend.data_ptr(), output.data_ptr()),
                   (m * k * 2, n * k // 2, scale.numel() * 2, addend.numel() * 2, m * n * 2),
                   _PARAMETERS(m, n, k, 1 if bias is not None else 0, 0), torch.cuda.current_stream(input.device).cuda_stream)
    return output


def _w4a16_linear_meta(input, packed_weight, scale, bias=None):
    del scale, bias
    return torch.empty((*input.shape[:-1], packed_weight.shape[0]), dtype=torch.float16, device="meta")


def register() -> None:
    """Defines `llmopt::w4a16_linear` (once) with a ROCm implementation and a meta kernel."""
    global _library, _native
    if _library is not None:
        return
    library = torch.library.Library("llmopt", "DEF")
    library.define("w4a16_linear(Tensor input, Tensor packed_weight, Tensor scale, Tensor? bias) -> Tensor")
    # what the native kernel of the above leaves to Python
    library.define("w4a16_linear_general(Tensor input, Tensor packed_weight, Tensor scale, Tensor? bias) -> Tensor")
    library.impl("w4a16_linear_general", _w4a16_linear_hip, "CUDA")  # ROCm tensors carry the CUDA dispatch key
    library.impl("w4a16_linear", _w4a16_linear_meta, "Meta")
    try:
        native = ctypes.CDLL(torch_library(torch.__version__))  # (its kernel registers itself as it is loaded)
        native.llmopt_torch_bind.argtypes = [ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p]
        native.llmopt_torch_bind.restype = None
    except OSError as error:
        warnings.warn(f"llmopt::w4a16_linear takes the longer way through Python ({error}); `python -m llmopt_amd.build` builds the other")
        native = None
        library.impl("w4a16_linear", _w4a16_linear_hip, "CUDA")
    _library, _native = library, native


register()
