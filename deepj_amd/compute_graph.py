"""Host-side lazy graph: the Python twin of the reference's
src/main/java/io/github/kirstenali/deepj/tensor/{ComputeGraph,GpuBuffer,GpuRuntime,TensorAdapters}.java.

It records ops as a flat int32 command stream, assigns buffer ids, batches
allocations and uploads, flushes everything through a GpuRuntime (five calls)
and releases buffers no tensor points at any more.  In a JVM deployment the
reference's own ComputeGraph plays this part unchanged; this twin exists so that
the native library can be driven and tested from Python with exactly the
protocol the Java class speaks (same encodings, same call order).
"""
from __future__ import annotations

import importlib.util
import os
import struct
import sys
import weakref
from typing import Protocol

import numpy as np

from . import opcodes as op
from .build import build_graph_core, graph_core_path



def _load_graph_core():
    name = __package__ + "._graph_core"
    if name not in sys.modules:
        path = graph_core_path()
        if not os.path.exists(path):            # not built yet
            build_graph_core()
        spec = importlib.util.spec_from_file_location(name, path)
        module = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(module)
        sys.modules[name] = module
    return sys.modules[name]


_graph_core = _load_graph_core()
GpuBuffer = _graph_core.GpuBuffer               # GpuBuffer.java:9-32


class GpuRuntime(Protocol):
    """GpuRuntime.java:9-28."""

    def allocBuffers(self, ids, sizes, count: int) -> None: ...
    def uploadBuffer(self, buf_id: int, data: np.ndarray) -> None: ...
    def downloadBuffer(self, buf_id: int, out: np.ndarray) -> None: ...
    def releaseBuffers(self, ids, count: int) -> None: ...
    def flushOps(self, cmd_stream: np.ndarray, length: int) -> None: ...


_pack_float, _unpack_int = struct.Struct("<f").pack, struct.Struct("<i").unpack


def float_bits(value: float) -> int:
    """Float.floatToRawIntBits as a signed int32."""
    try:
        return _unpack_int(_pack_float(value))[0]
    except OverflowError:                       # beyond fp32: infinity, as a cast gives
        return _unpack_int(_pack_float(np.float32(value)))[0]


# stride and buffer-id slots per opcode (ComputeGraph.java:89-147)
_OP_META: dict[int, tuple[int, tuple[int, ...]]] = {}
for _o in (op.OP_SQRT, op.OP_NEG, op.OP_EXP, op.OP_LOG, op.OP_TANH, op.OP_SIGMOID, op.OP_RELU, op.OP_GELU):
    _OP_META[_o] = (4, (1, 2))
for _o in (op.OP_ADD, op.OP_SUBTRACT, op.OP_MULTIPLY, op.OP_DIVIDE, op.OP_RELU_BACKWARD, op.OP_GELU_BACKWARD):
    _OP_META[_o] = (5, (1, 2, 3))
for _o in (op.OP_MULTIPLY_SCALAR, op.OP_ADD_SCALAR, op.OP_DIVIDE_SCALAR, op.OP_TRANSPOSE, op.OP_SUM_ROWS,
           op.OP_MEAN_ALONG_ROWS, op.OP_VARIANCE_ALONG_ROWS, op.OP_SUM_ALONG_ROWS, op.OP_MAX_ALONG_ROWS,
           op.OP_SOFTMAX_ROWS, op.OP_POW, op.OP_SUM_ABS, op.OP_SUM_SCALAR):
    _OP_META[_o] = (5, (1, 2))
_OP_META[op.OP_CLAMP] = (6, (1, 2))
for _o in (op.OP_SCATTER_ADD_ROWS, op.OP_SCATTER_ADD_ROWS_ATOMIC):
    _OP_META[_o] = (7, (1, 2, 3))
for _o in (op.OP_CROSS_ENTROPY_LOSS, op.OP_CROSS_ENTROPY_GRADIENT, op.OP_SOFTMAX_BACKWARD, op.OP_ADD_ROW_VECTOR,
           op.OP_ADD_BROADCAST_COLS, op.OP_SUBTRACT_BROADCAST_COLS, op.OP_DIVIDE_BROADCAST_COLS,
           op.OP_MULTIPLY_BROADCAST_ROWS, op.OP_MULTIPLY_BROADCAST_COLS):
    _OP_META[_o] = (6, (1, 2, 3))
_OP_META[op.OP_MATMUL] = (7, (1, 2, 3))
_OP_META[op.OP_LAYERNORM_BACKWARD] = (7, (1, 2, 3, 4))
_OP_META[op.OP_ADAMW_UPDATE] = (13, (1, 2, 3, 4))


class _OtherRef(weakref.ref):
    """A weak reference that remembers which buffer its object stood for."""
    __slots__ = ("id",)


class ComputeGraph(_graph_core.GraphCore):
    """ComputeGraph.java.  Buffer management (:172-234), flush (:528-671), materialize and release (:676-740) are
    csrc/graph_core.cpp, and so are the operations HipBackend records most; nothing walks all tracked tensors: buffers that may
    have lost their tensor announce themselves (a tensor that died, a replaced tag) and only those are looked at when a flush
    releases orphans.  The record* methods are the encodings (:238-518)."""

    def __init__(self, runtime: GpuRuntime):
        cls, calls = type(runtime), ()
        try:        # a runtime that only passes on to the native library says where its calls are; a class derived from it does not
            native = cls if "nativeCalls" in cls.__dict__ else None
            if native is not None:
                calls = cls.nativeCalls()
        except RuntimeError:                    # no library: the first call says so
            native = None
        super().__init__(runtime, getattr(runtime, "zeroBuffers", None),
                         getattr(runtime, "hostArray", None) or (lambda n: np.zeros(n, dtype=np.float32)), native, calls)

    # ── objects that stand in for a tensor: rows, cols, data, _data, _gpu_tag and setGpuTag are all that is asked of one ──
    def _ensureOther(self, o):
        if not hasattr(o, "_gpu_tag"):
            raise TypeError(f"expected a Tensor, not {type(o).__name__}")
        buf = o._gpu_tag
        if isinstance(buf, GpuBuffer):
            ref = (self._others or {}).get(buf.id)
            if ref is None or ref() is not o:
                self._trackOther(buf, o)
            if buf.needsUpload:
                self._uploadOther(buf, o, pack_f32(o))
                buf.needsUpload = buf.cpuStale = False
            return buf
        buf = _graph_core.GraphCore.newOutputBuffer(self, o.rows, o.cols)
        buf.cpuStale, buf.needsUpload = False, True
        self._uploadOther(buf, o, None if o._data is None else pack_f32(o))
        o.setGpuTag(buf)
        self._trackOther(buf, o)
        return buf

    def _trackOther(self, buf, o):
        self._forget(buf.id)
        if self._others is None:
            self._others = {}
        self._others[buf.id] = ref = _OtherRef(o, self._otherDied)
        ref.id = buf.id
        buf.graph = self

    def _otherDied(self, ref): self._lost(ref.id)

    def _uploadOther(self, buf, o, values):
        carrier = _tensor_class()(o.rows, o.cols)
        carrier._data = values
        self._upload(buf.id, carrier)

    def _downloadOther(self, buf, o):
        carrier = _tensor_class()(o.rows, o.cols)
        carrier._data = o._data
        self._download(buf, carrier)
        if o._data is not carrier._data:
            o._data = carrier._data

    def _bindOther(self, o, buf):
        o.setGpuTag(buf)
        self._trackOther(buf, o)

    def _materializeOther(self, o):
        if not hasattr(o, "_gpu_tag"):
            raise TypeError(f"expected a Tensor, not {type(o).__name__}")
        buf = o._gpu_tag
        if isinstance(buf, GpuBuffer) and buf.cpuStale:
            self.flush()
            self._downloadOther(buf, o)
            buf.cpuStale = False

    def _otherHolds(self, buf_id):
        o = self._others[buf_id]()
        return o is not None and isinstance(o._gpu_tag, GpuBuffer) and o._gpu_tag.id == buf_id

    def _releaseOthers(self):
        held = [o for o in (ref() for ref in self._others.values()) if o is not None]
        for o in held:
            buf = o._gpu_tag
            if isinstance(buf, GpuBuffer) and buf.cpuStale:
                self._downloadOther(buf, o)
                buf.cpuStale = buf.needsUpload = False
        for o in held:
            o.setGpuTag(None)
        return list(self._others)

    # ── op recording (ComputeGraph.java:238-518) ────────────────────────────
    def recordBinary(self, opcode, a, b, out): self._emit(opcode, a.id, b.id, out.id, out.floatCount())
    def recordMatmul(self, a, b, out, m, n, k): self._emit(op.OP_MATMUL, a.id, b.id, out.id, m, n, k)
    def recordUnary(self, opcode, inp, out): self._emit(opcode, inp.id, out.id, out.floatCount())

    def recordMultiplyScalar(self, inp, out, scalar):
        self._emit(op.OP_MULTIPLY_SCALAR, inp.id, out.id, float_bits(scalar), out.floatCount())

    def recordScalarUnary(self, opcode, inp, out, scalar):
        self._emit(opcode, inp.id, out.id, float_bits(scalar), out.floatCount())

    def recordPow(self, inp, out, exponent):
        self._emit(op.OP_POW, inp.id, out.id, float_bits(exponent), out.floatCount())

    def recordClamp(self, inp, out, lo, hi):
        self._emit(op.OP_CLAMP, inp.id, out.id, float_bits(lo), float_bits(hi), out.floatCount())

    def recordScatterAddRows(self, target, indices, grad, target_rows, target_cols, n_indices):
        self._emit(op.OP_SCATTER_ADD_ROWS, target.id, indices.id, grad.id, target_rows, target_cols, n_indices)

    def recordScatterAddRowsAtomic(self, target, indices, grad, target_rows, target_cols, n_indices):
        self._emit(op.OP_SCATTER_ADD_ROWS_ATOMIC, target.id, indices.id, grad.id, target_rows, target_cols, n_indices)

    def recordSumAbs(self, inp, out, rows, cols): self._emit(op.OP_SUM_ABS, inp.id, out.id, rows, cols)

    def recordCrossEntropyLoss(self, logits, targets, out, rows, cols):
        self._emit(op.OP_CROSS_ENTROPY_LOSS, logits.id, targets.id, out.id, rows, cols)

    def recordCrossEntropyGradient(self, logits, targets, out, rows, cols):
        self._emit(op.OP_CROSS_ENTROPY_GRADIENT, logits.id, targets.id, out.id, rows, cols)

    def recordSumScalar(self, inp, out, rows, cols): self._emit(op.OP_SUM_SCALAR, inp.id, out.id, rows, cols)
    def recordTranspose(self, inp, out, rows, cols): self._emit(op.OP_TRANSPOSE, inp.id, out.id, rows, cols)

    def recordRowBroadcast(self, opcode, a, row_vec, out, rows, cols):
        self._emit(opcode, a.id, row_vec.id, out.id, rows, cols)

    def recordColBroadcast(self, opcode, a, col_vec, out, rows, cols):
        self._emit(opcode, a.id, col_vec.id, out.id, rows, cols)

    def recordReduction(self, opcode, inp, out, rows, cols): self._emit(opcode, inp.id, out.id, rows, cols)
    def recordSoftmaxRows(self, inp, out, rows, cols): self._emit(op.OP_SOFTMAX_ROWS, inp.id, out.id, rows, cols)

    def recordSoftmaxBackward(self, grad, softmax, out, rows, cols):
        self._emit(op.OP_SOFTMAX_BACKWARD, grad.id, softmax.id, out.id, rows, cols)

    def recordLayerNormBackward(self, dxhat, xhat, std, out, rows, cols):
        self._emit(op.OP_LAYERNORM_BACKWARD, dxhat.id, xhat.id, std.id, out.id, rows, cols)

    def recordAdamWUpdate(self, w, g, mt, vt, lr, beta1, beta2, eps, weight_decay, bc1, bc2, n):
        self._emit(op.OP_ADAMW_UPDATE, w.id, g.id, mt.id, vt.id, float_bits(lr), float_bits(beta1),
                   float_bits(beta2), float_bits(eps), float_bits(weight_decay), float_bits(bc1), float_bits(bc2), n)


# What the operations of HipBackend record, through the graph's methods: csrc/graph_core.cpp does the same for tensors on a graph
# whose methods are ComputeGraph's, and calls these for everything else.
def _result(graph, out, into=None):
    return graph.createOutputTensor(out) if into is None else graph.bindTensorToBuffer(into, out)


def _binary(graph, opcode, name, a, b, in_place):
    if a.rows != b.rows or a.cols != b.cols:
        raise ValueError(f"Shape mismatch for {name}: {a.rows}x{a.cols} vs {b.rows}x{b.cols}")
    ga, gb = graph.ensureGpuBuffer(a), graph.ensureGpuBuffer(b)
    out = graph.newOutputBuffer(a.rows, a.cols)
    graph.recordBinary(opcode, ga, gb, out)
    return _result(graph, out, a if in_place else None)


def _unary(graph, opcode, a, in_place):
    ga = graph.ensureGpuBuffer(a)
    out = graph.newOutputBuffer(a.rows, a.cols)
    graph.recordUnary(opcode, ga, out)
    return _result(graph, out, a if in_place else None)


def _scalar(graph, opcode, a, value, in_place):
    ga = graph.ensureGpuBuffer(a)
    out = graph.newOutputBuffer(a.rows, a.cols)
    if opcode == op.OP_MULTIPLY_SCALAR:
        graph.recordMultiplyScalar(ga, out, value)
    elif opcode == op.OP_POW:
        graph.recordPow(ga, out, value)
    else:
        graph.recordScalarUnary(opcode, ga, out, value)
    return _result(graph, out, a if in_place else None)


_SHAPED = {op.OP_TRANSPOSE: "recordTranspose", op.OP_SOFTMAX_ROWS: "recordSoftmaxRows", op.OP_SUM_SCALAR: "recordSumScalar",
           op.OP_SUM_ABS: "recordSumAbs"}
_PAIRS = {op.OP_SOFTMAX_BACKWARD: "recordSoftmaxBackward", op.OP_CROSS_ENTROPY_GRADIENT: "recordCrossEntropyGradient"}


def _shaped(graph, opcode, a, rows, cols):
    ga = graph.ensureGpuBuffer(a)
    out = graph.newOutputBuffer(rows, cols)
    if opcode in _SHAPED:
        getattr(graph, _SHAPED[opcode])(ga, out, a.rows, a.cols)
    else:
        graph.recordReduction(opcode, ga, out, a.rows, a.cols)
    return _result(graph, out)


def _pair(graph, opcode, a, b):
    ga, gb = graph.ensureGpuBuffer(a), graph.ensureGpuBuffer(b)
    out = graph.newOutputBuffer(a.rows, a.cols)
    getattr(graph, _PAIRS[opcode])(ga, gb, out, a.rows, a.cols)
    return _result(graph, out)


def _row_broadcast(graph, opcode, a, v):
    if v.rows != 1 or v.cols != a.cols:
        raise ValueError(f"Expected row vector 1x{a.cols} but got {v.rows}x{v.cols}")
    ga, gv = graph.ensureGpuBuffer(a), graph.ensureGpuBuffer(v)
    out = graph.newOutputBuffer(a.rows, a.cols)
    graph.recordRowBroadcast(opcode, ga, gv, out, a.rows, a.cols)
    return _result(graph, out)


def _col_broadcast(graph, opcode, a, v):
    if v.rows != a.rows or v.cols != 1:
        raise ValueError(f"Expected col vector {a.rows}x1 but got {v.rows}x{v.cols}")
    ga, gv = graph.ensureGpuBuffer(a), graph.ensureGpuBuffer(v)
    out = graph.newOutputBuffer(a.rows, a.cols)
    graph.recordColBroadcast(opcode, ga, gv, out, a.rows, a.cols)
    return _result(graph, out)


def _matmul(graph, opcode, a, b):
    if a.cols != b.rows:
        raise ValueError(f"Shape mismatch for matmul: {a.rows}x{a.cols} vs {b.rows}x{b.cols}")
    ga, gb = graph.ensureGpuBuffer(a), graph.ensureGpuBuffer(b)
    out = graph.newOutputBuffer(a.rows, b.cols)
    graph.recordMatmul(ga, gb, out, a.rows, b.cols, a.cols)
    return _result(graph, out)


def _adamw(graph, opcode, w, g, mt, vt, lr, beta1, beta2, eps, weight_decay, bc1, bc2):
    gw, gg, gm, gv = (graph.ensureGpuBuffer(t) for t in (w, g, mt, vt))
    graph.recordAdamWUpdate(gw, gg, gm, gv, lr, beta1, beta2, eps, weight_decay, bc1, bc2, w.rows * w.cols)
    for b in (gw, gm, gv):
        b.cpuStale = True
        b.needsUpload = False


_graph_core.set_methods(
    {"binary": _binary, "unary": _unary, "scalar": _scalar, "shaped": _shaped, "pair": _pair, "rowBroadcast": _row_broadcast,
     "colBroadcast": _col_broadcast, "matmul": _matmul, "adamW": _adamw}, ComputeGraph,
    ["ensureGpuBuffer", "newOutputBuffer", "createOutputTensor", "bindTensorToBuffer", "tensorLetGo", "flush", "_emit", "recordBinary", "recordUnary",
     "recordMultiplyScalar", "recordPow", "recordScalarUnary", "recordReduction", "recordRowBroadcast", "recordColBroadcast", "recordMatmul",
     "recordAdamWUpdate", *_SHAPED.values(), *_PAIRS.values()])


def _tensor_class():
    from .tensor import Tensor
    return Tensor


# TensorAdapters.java:9-47
def pack_f32(t) -> np.ndarray:
    return t.data.astype(np.float32, order="C").reshape(-1)          # a copy: the tensor may change before the flush


def unpack_f32_into(src: np.ndarray, dst) -> None:
    if src.size != dst.rows * dst.cols:
        raise ValueError(f"Size mismatch: src has {src.size} floats but tensor is {dst.rows}x{dst.cols}")
    if dst.data.flags.writeable:
        dst.data[...] = np.reshape(src, (dst.rows, dst.cols))
    else:
        dst._data = np.reshape(src, (dst.rows, dst.cols)).astype(np.float32, copy=False)


def from_int_column(values) -> "object":
    t = _tensor_class()(len(values), 1)
    t.data[:, 0] = np.asarray(values, dtype=np.float32)
    return t


_graph_core.set_helpers(np.empty, np.zeros, np.float32, pack_f32, unpack_f32_into, _OP_META, op.OP_FILL)
