"""HipBackend: the TensorBackend of this library, a structural twin of the reference's
MetalBackend (src/main/java/io/github/kirstenali/deepj/tensor/metal/MetalBackend.java:8-633):
every op is recorded into a private ComputeGraph and nothing runs until a tensor is
materialised.  In-place ops get a new output buffer and rebind the tensor
(MetalBackend.java:400-411); ops that return a scalar materialise at once
(:247-266,541-555); integer targets and indices travel as float column tensors (:43-54).

HipGpuRuntime is the five-call pass-through to the native library
(cf. MetalGpuRuntime.java:9-35).
"""
from __future__ import annotations

import numpy as np

from . import opcodes as op
from ._native import HipNative, call_addresses, host_array
from .compute_graph import ComputeGraph, GpuBuffer, _graph_core as record
from .tensor import Tensor


class HipGpuRuntime:
    """Five calls passed on to the native library; a graph over an object of exactly this class makes them itself, as long as
    nothing is put in place of them or of HipNative's."""

    nativeCalls = staticmethod(call_addresses)

    def allocBuffers(self, ids, sizes, count): HipNative.nativeAllocBuffers(ids, sizes, count)
    def uploadBuffer(self, buf_id, data): HipNative.nativeUploadBuffer(buf_id, data)
    def downloadBuffer(self, buf_id, out): HipNative.nativeDownloadBuffer(buf_id, out)
    def releaseBuffers(self, ids, count): HipNative.nativeReleaseBuffers(ids, count)
    def flushOps(self, cmd_stream, length): HipNative.nativeFlushOps(cmd_stream if len(cmd_stream) == length else cmd_stream[:length], length)
    def hostArray(self, n): return host_array(n)

    def zeroBuffers(self, buffers):
        cmd = [w for buf_id, n in buffers for w in (op.OP_FILL, buf_id, 0, n)]
        HipNative.nativeFlushOps(cmd, len(cmd))


record.set_native(HipGpuRuntime, ("allocBuffers", "uploadBuffer", "downloadBuffer", "releaseBuffers", "flushOps", "zeroBuffers"),
                  HipNative, ("nativeAllocBuffers", "nativeUploadBuffer", "nativeDownloadBuffer", "nativeReleaseBuffers", "nativeFlushOps"))


class HipBackend:
    def __init__(self, runtime=None):
        self.graph = ComputeGraph(runtime if runtime is not None else HipGpuRuntime())
        self._int_column_scratch: dict[int, Tensor] = {}

    # ── lazy helpers ────────────────────────────────────────────────────────
    def _in(self, t): return self.graph.ensureGpuBuffer(t)
    def _out(self, buf): return self.graph.createOutputTensor(buf)

    def _int_column(self, values) -> Tensor:
        t = self._int_column_scratch.get(len(values))
        if t is None:
            t = Tensor(len(values), 1)
            self._int_column_scratch[len(values)] = t
        t.data[:, 0] = np.asarray(values, dtype=np.float32)
        if isinstance(t.getGpuTag(), GpuBuffer):
            t.getGpuTag().needsUpload = True
            t.getGpuTag().cpuStale = False
        return t

    def materializeTensor(self, t): self.graph.materialize(t)

    def releaseResources(self):
        self.graph.releaseAll()
        self._int_column_scratch.clear()

    # ── matmul / element-wise ───────────────────────────────────────────────
    def matmul(self, a, b): return record.matmul(self.graph, op.OP_MATMUL, a, b)
    def add(self, a, b): return record.binary(self.graph, op.OP_ADD, "add", a, b, False)
    def subtract(self, a, b): return record.binary(self.graph, op.OP_SUBTRACT, "subtract", a, b, False)
    def multiply(self, a, b): return record.binary(self.graph, op.OP_MULTIPLY, "multiply", a, b, False)
    def divide(self, a, b): return record.binary(self.graph, op.OP_DIVIDE, "divide", a, b, False)
    def reluBackward(self, x, g): return record.binary(self.graph, op.OP_RELU_BACKWARD, "reluBackward", x, g, False)
    def geluBackward(self, x, g): return record.binary(self.graph, op.OP_GELU_BACKWARD, "geluBackward", x, g, False)

    # ── broadcasts ──────────────────────────────────────────────────────────
    def addRowVector(self, a, v): return record.rowBroadcast(self.graph, op.OP_ADD_ROW_VECTOR, a, v)
    def addBroadcastRows(self, a, v): return self.addRowVector(a, v)
    def multiplyBroadcastRows(self, a, v): return record.rowBroadcast(self.graph, op.OP_MULTIPLY_BROADCAST_ROWS, a, v)
    def addBroadcastCols(self, a, v): return record.colBroadcast(self.graph, op.OP_ADD_BROADCAST_COLS, a, v)
    def subtractBroadcastCols(self, a, v): return record.colBroadcast(self.graph, op.OP_SUBTRACT_BROADCAST_COLS, a, v)
    def divideBroadcastCols(self, a, v): return record.colBroadcast(self.graph, op.OP_DIVIDE_BROADCAST_COLS, a, v)
    def multiplyBroadcastCols(self, a, v): return record.colBroadcast(self.graph, op.OP_MULTIPLY_BROADCAST_COLS, a, v)

    # ── scalar ops ──────────────────────────────────────────────────────────
    def multiplyScalar(self, a, s): return record.scalar(self.graph, op.OP_MULTIPLY_SCALAR, a, s, False)
    def addScalar(self, a, s): return record.scalar(self.graph, op.OP_ADD_SCALAR, a, s, False)
    def divideScalar(self, a, s): return record.scalar(self.graph, op.OP_DIVIDE_SCALAR, a, s, False)

    # ── reductions ──────────────────────────────────────────────────────────
    def sumRows(self, a): return record.shaped(self.graph, op.OP_SUM_ROWS, a, 1, a.cols)
    def sumAlongCols(self, a): return self.sumRows(a)
    def sumAlongRows(self, a): return record.shaped(self.graph, op.OP_SUM_ALONG_ROWS, a, a.rows, 1)
    def meanAlongRows(self, a): return record.shaped(self.graph, op.OP_MEAN_ALONG_ROWS, a, a.rows, 1)
    def varianceAlongRows(self, a): return record.shaped(self.graph, op.OP_VARIANCE_ALONG_ROWS, a, a.rows, 1)
    def maxAlongRows(self, a): return record.shaped(self.graph, op.OP_MAX_ALONG_ROWS, a, a.rows, 1)

    def sum(self, a) -> float:
        scalar = record.shaped(self.graph, op.OP_SUM_SCALAR, a, 1, 1)
        scalar.materialize()
        return float(scalar.data[0, 0])

    def sumAbs(self, a) -> float:
        scalar = self.sumRows(record.shaped(self.graph, op.OP_SUM_ABS, a, a.rows, 1))
        scalar.materialize()
        return float(scalar.data[0, 0])

    # ── unary ───────────────────────────────────────────────────────────────
    def transpose(self, a): return record.shaped(self.graph, op.OP_TRANSPOSE, a, a.cols, a.rows)

    def clamp(self, a, lo, hi):
        ga = self._in(a)
        out = self.graph.newOutputBuffer(a.rows, a.cols)
        self.graph.recordClamp(ga, out, lo, hi)
        return self._out(out)

    def pow(self, a, exponent): return record.scalar(self.graph, op.OP_POW, a, exponent, False)
    def sqrt(self, a): return record.unary(self.graph, op.OP_SQRT, a, False)
    def neg(self, a): return record.unary(self.graph, op.OP_NEG, a, False)
    def exp(self, a): return record.unary(self.graph, op.OP_EXP, a, False)
    def log(self, a): return record.unary(self.graph, op.OP_LOG, a, False)
    def tanh(self, a): return record.unary(self.graph, op.OP_TANH, a, False)
    def sigmoid(self, a): return record.unary(self.graph, op.OP_SIGMOID, a, False)
    def relu(self, a): return record.unary(self.graph, op.OP_RELU, a, False)
    def gelu(self, a): return record.unary(self.graph, op.OP_GELU, a, False)

    # ── softmax ─────────────────────────────────────────────────────────────
    def softmaxRows(self, logits): return record.shaped(self.graph, op.OP_SOFTMAX_ROWS, logits, logits.rows, logits.cols)

    def softmaxBackward(self, grad, softmax):
        Tensor.requireSameShape(grad, softmax, "softmaxBackward")
        return record.pair(self.graph, op.OP_SOFTMAX_BACKWARD, grad, softmax)

    # ── in-place: new buffer, rebind (MetalBackend.java:400-526) ────────────
    def addInPlace(self, a, b): record.binary(self.graph, op.OP_ADD, "addInPlace", a, b, True)
    def subtractInPlace(self, a, b): record.binary(self.graph, op.OP_SUBTRACT, "subtractInPlace", a, b, True)
    def multiplyInPlace(self, a, b): record.binary(self.graph, op.OP_MULTIPLY, "multiplyInPlace", a, b, True)
    def divideInPlace(self, a, b): record.binary(self.graph, op.OP_DIVIDE, "divideInPlace", a, b, True)
    def multiplyScalarInPlace(self, a, s): record.scalar(self.graph, op.OP_MULTIPLY_SCALAR, a, s, True)
    def addScalarInPlace(self, a, s): record.scalar(self.graph, op.OP_ADD_SCALAR, a, s, True)
    def divideScalarInPlace(self, a, s): record.scalar(self.graph, op.OP_DIVIDE_SCALAR, a, s, True)
    def sqrtInPlace(self, a): record.unary(self.graph, op.OP_SQRT, a, True)
    def negInPlace(self, a): record.unary(self.graph, op.OP_NEG, a, True)
    def expInPlace(self, a): record.unary(self.graph, op.OP_EXP, a, True)
    def logInPlace(self, a): record.unary(self.graph, op.OP_LOG, a, True)
    def reluInPlace(self, a): record.unary(self.graph, op.OP_RELU, a, True)
    def geluInPlace(self, a): record.unary(self.graph, op.OP_GELU, a, True)
    def tanhInPlace(self, a): record.unary(self.graph, op.OP_TANH, a, True)
    def sigmoidInPlace(self, a): record.unary(self.graph, op.OP_SIGMOID, a, True)

    # ── fused ops ───────────────────────────────────────────────────────────
    def crossEntropyGradient(self, logits, targets):
        Tensor.requireTargetsMatchRows(logits, targets)
        return record.pair(self.graph, op.OP_CROSS_ENTROPY_GRADIENT, logits, self._int_column(targets))

    def crossEntropyLoss(self, logits, targets) -> float:
        Tensor.requireTargetsMatchRows(logits, targets)
        tt = self._int_column(targets)
        gl, gt = self._in(logits), self._in(tt)
        rows = self.graph.newOutputBuffer(logits.rows, 1)
        self.graph.recordCrossEntropyLoss(gl, gt, rows, logits.rows, logits.cols)
        scalar = self.sumRows(self._out(rows)).divideScalar(logits.rows)
        scalar.materialize()
        return float(scalar.data[0, 0])

    def adamWUpdate(self, w, g, mt, vt, lr, beta1, beta2, eps, weight_decay, bc1, bc2):
        for other in (g, mt, vt):
            Tensor.requireSameShape(w, other, "adamWUpdate")
        record.adamW(self.graph, op.OP_ADAMW_UPDATE, w, g, mt, vt, lr, beta1, beta2, eps, weight_decay, bc1, bc2)

    def layerNormBackward(self, dxhat, xhat, std, dim):
        Tensor.requireSameShape(dxhat, xhat, "layerNormBackward")
        if dim != dxhat.cols:
            raise ValueError(f"layerNormBackward: dim={dim} must equal tensor cols={dxhat.cols}")
        if std.rows != dxhat.rows or std.cols != 1:
            raise ValueError(f"layerNormBackward: std must be {dxhat.rows}x1 but got {std.rows}x{std.cols}")
        gd, gx, gs = self._in(dxhat), self._in(xhat), self._in(std)
        out = self.graph.newOutputBuffer(dxhat.rows, dxhat.cols)
        self.graph.recordLayerNormBackward(gd, gx, gs, out, dxhat.rows, dxhat.cols)
        return self._out(out)

    def scatterAddRows(self, target, indices, grad):
        if len(indices) != grad.rows:
            raise ValueError(f"scatterAddRows: indices length {len(indices)} must match grad rows {grad.rows}")
        if target.cols != grad.cols:
            raise ValueError(f"scatterAddRows: target cols {target.cols} must match grad cols {grad.cols}")
        if len(indices) == 0:
            return
        it = self._int_column(indices)
        gt, gg, gi = self._in(target), self._in(grad), self._in(it)
        self.graph.recordScatterAddRowsAtomic(gt, gi, gg, target.rows, target.cols, len(indices))
        gt.cpuStale = True
        gt.needsUpload = False
