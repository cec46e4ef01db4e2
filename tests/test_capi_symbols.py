"""The C-ABI library loads without a GPU and exports every function include/deepj_hip.h declares;
compute entry points fail loudly (no CPU fallback) when no device is present."""
import ctypes
import os
import re

import numpy as np
import pytest

from deepj_amd import HipNative, LIB_PATH

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_functions():
    text = open(os.path.join(ROOT, "include", "deepj_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(deepj_(?:hip|runner|host)_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    lib = ctypes.CDLL(LIB_PATH)
    names = declared_functions()
    assert "deepj_hip_flush_ops" in names and len(names) >= 12
    missing = [n for n in names if not hasattr(lib, n)]
    assert not missing, missing


def test_opcode_numbers_match_header():
    from deepj_amd import opcodes
    text = open(os.path.join(ROOT, "include", "deepj_hip.h")).read()
    for name, value in re.findall(r"DJ_(OP_[A-Z0-9_]+)\s*=\s*(\d+)", text):
        assert getattr(opcodes, name) == int(value), name


@pytest.mark.skipif(os.path.exists("/dev/kfd"), reason="checks the no-GPU failure path")
def test_no_silent_cpu_fallback_without_a_device():
    with pytest.raises(RuntimeError, match="no HIP device"):
        HipNative.nativeAllocBuffers([0], [4], 1)
    with pytest.raises(RuntimeError):
        HipNative.nativeFlushOps(np.array([1, 0, 0, 0, 4], dtype=np.int32), 5)
    assert HipNative.q8Floats(64, 2) == (256 + 2 * 2 * 4) // 4      # pure size arithmetic needs no device


def test_a_finaliser_keeps_the_message_of_a_failed_call():
    """Arrays over the library's host memory give their block back whenever they are collected, also between a failed call
    and the reading of its message."""
    lib = ctypes.CDLL(LIB_PATH)
    lib.deepj_hip_last_error.restype = ctypes.c_char_p
    lib.deepj_hip_host_free.argtypes = [ctypes.c_void_p]
    lib.deepj_hip_host_free.restype = None
    other = ctypes.create_string_buffer(64)                          # no block of the library: ignored
    assert lib.deepj_hip_upload(1 << 30, other, ctypes.c_int64(1)) != 0
    message = lib.deepj_hip_last_error()
    assert message
    lib.deepj_hip_host_free(ctypes.addressof(other))
    assert lib.deepj_hip_last_error() == message


def test_device_code_is_built_for_gfx950_with_the_required_flags():
    """Every HIP source is compiled for gfx950 with packed-FP32 instructions switched off and with the leading
    kernel arguments preloaded into registers (the decode kernels' argument order relies on it)."""
    from deepj_amd import build
    assert build.ARCH == "gfx950"
    flags = " ".join(build.COMMON)
    assert "-Xclang -target-feature -Xclang -packed-fp32-ops" in flags
    assert "-mllvm -amdgpu-kernarg-preload-count=16" in flags
    assert all(os.path.exists(os.path.join(build.CSRC, src)) for src in build.SOURCES)
    # the device pass honours the flag (the host pass only notes that it does not know the feature): a float2 probe
    # kernel compiled with it holds no v_pk_*_f32 instruction, and holds one without it
    build.verify_packed_fp32_off()
