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

import array
import struct
import weakref
from typing import Protocol

import numpy as np

from . import opcodes as op


class GpuRuntime(Protocol):
    """GpuRuntime.java:9-28."""

    def allocBuffers(self, ids, sizes, count: int) -> None: ...
    def uploadBuffer(self, buf_id: int, data: np.ndarray) -> None: ...
    def downloadBuffer(self, buf_id: int, out: np.ndarray) -> None: ...
    def releaseBuffers(self, ids, count: int) -> None: ...
    def flushOps(self, cmd_stream: np.ndarray, length: int) -> None: ...


class GpuBuffer:
    """GpuBuffer.java:9-32."""

    __slots__ = ("id", "rows", "cols", "needsUpload", "cpuStale", "allocatedOnGpu", "graph")

    def __init__(self, id: int, rows: int, cols: int, needs_upload: bool, graph=None):
        self.id, self.rows, self.cols = id, rows, cols
        self.needsUpload = needs_upload
        self.cpuStale = False
        self.allocatedOnGpu = True
        self.graph = graph          # the graph that tracks it: told when a tensor lets go of this buffer

    def floatCount(self) -> int:
        return self.rows * self.cols


_pack_float, _unpack_int = struct.Struct("<f").pack, struct.Struct("<i").unpack


def float_bits(value: float) -> int:
    """Float.floatToRawIntBits as a signed int32."""
    try:
        return _unpack_int(_pack_float(value))[0]
    except OverflowError:                       # beyond fp32: infinity, as a cast gives
        return _unpack_int(_pack_float(np.float32(value)))[0]


class _TensorRef(weakref.ref):
    """A weak reference that remembers which buffer its tensor stood for."""
    __slots__ = ("id",)


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


class ComputeGraph:
    """Recording one op costs a few microseconds of host time, as much as its launch, so nothing here walks all tracked
    tensors: buffers that may have lost their tensor announce themselves (a dead weak reference, a replaced tag) and only
    those are looked at when a flush releases orphans."""

    def __init__(self, runtime: GpuRuntime):
        if runtime is None:
            raise TypeError("runtime")          # Objects.requireNonNull
        self.runtime = runtime
        self._next_buf_id = 0
        self._cmd = array.array("i")
        self._op_count = 0
        self._pending_allocs: list[GpuBuffer] = []
        self._pending_uploads: list[tuple[int, np.ndarray | int]] = []      # values, or how many zeros
        self._buf_to_tensor: dict[int, _TensorRef] = {}
        self._maybe_orphans: list[int] = []
        self._zero_buffers = getattr(runtime, "zeroBuffers", None)
        self._host_array = getattr(runtime, "hostArray", None) or (lambda n: np.zeros(n, dtype=np.float32))

    # ── buffer management (ComputeGraph.java:172-234) ───────────────────────
    def ensureGpuBuffer(self, t) -> GpuBuffer:
        existing = t._gpu_tag
        if isinstance(existing, GpuBuffer):
            ref = self._buf_to_tensor.get(existing.id)
            if ref is None or ref() is not t:
                self._track(existing, t)
            if existing.needsUpload:
                self._pending_uploads.append((existing.id, pack_f32(t)))
                existing.needsUpload = False
                existing.cpuStale = False
            return existing
        buf = GpuBuffer(self._next_buf_id, t.rows, t.cols, True, self)
        self._next_buf_id += 1
        buf.allocatedOnGpu = False
        self._pending_allocs.append(buf)
        # a tensor nothing was ever written to is cleared on the device, where the runtime can, instead of sending zeros
        zeros = t._data is None and self._zero_buffers is not None
        self._pending_uploads.append((buf.id, buf.rows * buf.cols if zeros else pack_f32(t)))
        t.setGpuTag(buf)
        self._track(buf, t)
        return buf

    def _track(self, buf: GpuBuffer, t) -> None:
        ref = _TensorRef(t, self._tensor_died)
        ref.id = buf.id
        self._buf_to_tensor[buf.id] = ref
        buf.graph = self

    def _tensor_died(self, ref) -> None:
        self._maybe_orphans.append(ref.id)

    def tensorLetGo(self, buf: GpuBuffer) -> None:
        """Tensor.setGpuTag: `buf` is no longer the tag of a tensor that had it."""
        self._maybe_orphans.append(buf.id)

    def newOutputBuffer(self, rows: int, cols: int) -> GpuBuffer:
        buf = GpuBuffer(self._next_buf_id, rows, cols, False, self)
        self._next_buf_id += 1
        buf.cpuStale = True
        buf.allocatedOnGpu = False
        self._pending_allocs.append(buf)
        return buf

    def createOutputTensor(self, buf: GpuBuffer):
        t = _tensor_class()(buf.rows, buf.cols)
        t._gpu_tag = buf
        self._track(buf, t)
        return t

    def bindTensorToBuffer(self, t, buf: GpuBuffer) -> None:
        t.setGpuTag(buf)
        self._track(buf, t)

    # ── op recording (ComputeGraph.java:238-518) ────────────────────────────
    def _emit(self, *words: int) -> None:
        self._cmd.extend(words)
        self._op_count += 1

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

    def isEmpty(self) -> bool:
        return self._op_count == 0

    # ── flush (ComputeGraph.java:528-671) ───────────────────────────────────
    def flush(self) -> None:
        if self._op_count == 0 and not self._pending_allocs:
            self._release_orphans()
            return
        self._allocate_pending()
        self._upload_pending()
        self._execute_pending()
        self._release_orphans()

    def _allocate_pending(self) -> None:
        pending = self._pending_allocs
        if not pending:
            return
        self.runtime.allocBuffers(array.array("i", [b.id for b in pending]), array.array("i", [b.rows * b.cols for b in pending]), len(pending))
        for b in pending:
            b.allocatedOnGpu = True
        self._pending_allocs = []

    def _upload_pending(self) -> None:
        zeros = [u for u in self._pending_uploads if type(u[1]) is int]
        if zeros:                               # first: a buffer's zeros come before whatever else is sent to it
            self._zero_buffers(zeros)
        for buf_id, data in self._pending_uploads:
            if type(data) is not int:
                self.runtime.uploadBuffer(buf_id, data)
        self._pending_uploads.clear()

    def _execute_pending(self) -> None:
        if self._op_count > 0:
            self.runtime.flushOps(self._cmd, len(self._cmd))        # (fails before its first launch: the ops stay recorded)
        self._cmd, self._op_count = array.array("i"), 0

    def _release_orphans(self) -> None:
        if not self._maybe_orphans:
            return
        candidates, self._maybe_orphans = self._maybe_orphans, []
        orphans = []
        for buf_id in dict.fromkeys(candidates):
            ref = self._buf_to_tensor.get(buf_id)
            if ref is None:
                continue
            t = ref()
            if t is not None and isinstance(t._gpu_tag, GpuBuffer) and t._gpu_tag.id == buf_id:
                continue
            if self._op_count > 0 and self._referenced_by_pending_ops(buf_id):
                self._maybe_orphans.append(buf_id)
                continue
            orphans.append(buf_id)
            del self._buf_to_tensor[buf_id]
        if not orphans:
            return
        if self._pending_allocs or self._pending_uploads:
            gone = set(orphans)
            self._pending_allocs = [b for b in self._pending_allocs if b.id not in gone]
            self._pending_uploads = [u for u in self._pending_uploads if u[0] not in gone]
        self.runtime.releaseBuffers(array.array("i", orphans), len(orphans))

    def _referenced_by_pending_ops(self, buf_id: int) -> bool:
        pos = 0
        while pos < len(self._cmd):
            meta = _OP_META.get(self._cmd[pos])
            if meta is None:
                return True                     # unknown op: be conservative
            stride, slots = meta
            if any(self._cmd[pos + s] == buf_id for s in slots):
                return True
            pos += stride
        return False

    # ── materialize / release (ComputeGraph.java:676-740) ───────────────────
    def materialize(self, t) -> None:
        buf = t._gpu_tag
        if not isinstance(buf, GpuBuffer) or not buf.cpuStale:
            return
        self.flush()
        self._download(buf, t)
        buf.cpuStale = False

    def _download(self, buf: GpuBuffer, t) -> None:
        """The buffer's values in the tensor's host array: written there directly, and into an array of the runtime's
        own kind where the tensor has none yet."""
        data = t._data
        if data is None or not data.flags.c_contiguous or data.dtype != np.float32:
            flat = self._host_array(buf.rows * buf.cols)
            self.runtime.downloadBuffer(buf.id, flat)
            if data is None and flat.size == t.rows * t.cols:
                t._data = flat.reshape(t.rows, t.cols)
            else:
                unpack_f32_into(flat, t)
            return
        if data.size != buf.rows * buf.cols:
            raise ValueError(f"Size mismatch: src has {buf.rows * buf.cols} floats but tensor is {t.rows}x{t.cols}")
        self.runtime.downloadBuffer(buf.id, data.reshape(-1))

    def releaseAll(self) -> None:
        self.flush()
        for ref in list(self._buf_to_tensor.values()):
            t = ref()
            if t is None:
                continue
            gb = t._gpu_tag
            if not isinstance(gb, GpuBuffer) or not gb.cpuStale:
                continue
            self._download(gb, t)
            gb.cpuStale = False
            gb.needsUpload = False
        for ref in self._buf_to_tensor.values():
            t = ref()
            if t is not None:
                t.setGpuTag(None)
        if self._buf_to_tensor:
            ids = array.array("i", self._buf_to_tensor.keys())
            self.runtime.releaseBuffers(ids, len(ids))
        self._buf_to_tensor.clear()
        self._maybe_orphans.clear()
        self._pending_allocs = []
        self._pending_uploads.clear()
        self._cmd, self._op_count = array.array("i"), 0
        self._next_buf_id = 0


_tensor_type = None


def _tensor_class():
    global _tensor_type
    if _tensor_type is None:
        from .tensor import Tensor
        _tensor_type = Tensor
    return _tensor_type


# TensorAdapters.java:9-47
def pack_f32(t) -> np.ndarray:
    return t.data.astype(np.float32, order="C").reshape(-1)          # a copy: the tensor may change before the flush


def unpack_f32_into(src: np.ndarray, dst) -> None:
    if src.size != dst.rows * dst.cols:
        raise ValueError(f"Size mismatch: src has {src.size} floats but tensor is {dst.rows}x{dst.cols}")
    dst.data.reshape(-1)[:] = src


def from_int_column(values) -> "object":
    from .tensor import Tensor
    t = Tensor(len(values), 1)
    t.data[:, 0] = np.asarray(values, dtype=np.float32)
    return t
