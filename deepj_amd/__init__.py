"""deepj_amd: MI355X (gfx950) backend for DeepJ behind its TensorBackend / ComputeGraph /
GpuRuntime boundary.  The compute lives in libdeepj_hip.so (hand-written HIP kernels
reached through the C ABI in include/deepj_hip.h); this package is the host-side twin of
the reference's Java classes around that boundary."""
import importlib

from . import opcodes
from ._native import HipNative, LIB_PATH
from .models import (DeepSeekConfig, DeepSeekModel, GPTConfig, GPTModel, JavaRandom, LlamaConfig, LlamaModel,
                     TextGenerator)
from .persistence import ModelSerializer, parameter_names, parameter_shapes

__all__ = ["ModelSerializer", "parameter_names", "parameter_shapes", "opcodes", "HipNative", "LIB_PATH", "ComputeGraph", "GpuBuffer", "HipBackend", "HipGpuRuntime", "Tensor",
           "LlamaConfig", "LlamaModel", "GPTConfig", "GPTModel", "DeepSeekConfig", "DeepSeekModel", "TextGenerator", "JavaRandom"]

# The tensor side is loaded when it is first asked for: models need nothing of it, nor its extension (csrc/graph_core.cpp).
_TENSOR_SIDE = {"ComputeGraph": "compute_graph", "GpuBuffer": "compute_graph", "HipBackend": "hip_backend", "HipGpuRuntime": "hip_backend",
                "Tensor": "tensor"}


def __getattr__(name):
    if name in _TENSOR_SIDE.values():
        return importlib.import_module("." + name, __name__)
    if name in _TENSOR_SIDE:
        globals()[name] = value = getattr(importlib.import_module("." + _TENSOR_SIDE[name], __name__), name)
        return value
    raise AttributeError(f"module {__name__!r} has no attribute {name!r}")


def __dir__(): return sorted({*globals(), *_TENSOR_SIDE, *_TENSOR_SIDE.values()})
