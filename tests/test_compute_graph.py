"""The lazy-graph protocol without a GPU: a recording GpuRuntime logs the five calls, as the
reference's own src/test/java/io/github/kirstenali/deepj/tensor/ComputeGraphTest.java:546-591
does.  Each test cites the reference test it mirrors."""
import ctypes as C
import gc
import struct
import subprocess
import threading
import time
import weakref

import numpy as np
import pytest

from deepj_amd import ComputeGraph, GpuBuffer, HipBackend, HipGpuRuntime, HipNative, Tensor, opcodes as op


class RecordingRuntime:
    def __init__(self):
        self.allocCalls, self.uploads, self.downloads, self.flushCalls, self.releaseCalls = [], [], [], [], []
        self.downloadResult = None

    def allocBuffers(self, ids, sizes, count):
        self.allocCalls.append((np.array(ids).copy(), np.array(sizes).copy(), count))

    def uploadBuffer(self, buf_id, data):
        self.uploads.append((buf_id, np.array(data).copy()))

    def downloadBuffer(self, buf_id, out):
        self.downloads.append(buf_id)
        if self.downloadResult is not None:
            n = min(len(self.downloadResult), out.size)
            out[:n] = self.downloadResult[:n]

    def releaseBuffers(self, ids, count):
        self.releaseCalls.append((np.array(ids).copy(), count))

    def flushOps(self, cmd, length):
        self.flushCalls.append((np.array(cmd[:length]).copy(), length))


class NativeLibrary:
    """The five calls and the error text as C functions, which a graph calls by address: what a library does with ids and sizes, the
    calls in order, and one upload that fails when told to."""

    def __init__(self):
        ids, values = C.POINTER(C.c_int32), C.POINTER(C.c_float)
        self.calls, self.sizes, self.held, self.fail_upload, self.during = [], {}, {}, False, None
        self.message = C.create_string_buffer(b"the library says so")
        self.functions = [C.CFUNCTYPE(C.c_int, ids, ids, C.c_int32)(self.alloc), C.CFUNCTYPE(C.c_int, C.c_int32, values, C.c_int64)(self.upload),
                          C.CFUNCTYPE(C.c_int, C.c_int32, values, C.c_int64)(self.download), C.CFUNCTYPE(C.c_int, ids, C.c_int32)(self.release),
                          C.CFUNCTYPE(C.c_int, ids, C.c_int32)(self.flush), C.CFUNCTYPE(C.c_void_p)(lambda: C.addressof(self.message))]

    def graph(self):
        class Runtime:
            nativeCalls = staticmethod(lambda: tuple(C.cast(f, C.c_void_p).value for f in self.functions))
            def zeroBuffers(self, buffers): raise AssertionError("not called where the library is")
            def hostArray(self, n): return np.empty(n, np.float32)
        return ComputeGraph(Runtime())

    def log(self, name, *args):
        self.calls.append((name, *args))
        if self.during:
            self.during(name)

    def alloc(self, ids, sizes, n):
        self.log("alloc", ids[:n])
        for i, size in zip(ids[:n], sizes[:n]):
            self.sizes.setdefault(i, size)                            # (an id that exists stays as it is)
        return 0

    def upload(self, i, values, n):
        self.log("upload", i, n)
        if self.fail_upload or n > self.sizes.get(i, -1):
            return 1
        self.held[i] = values[:n]
        return 0

    def download(self, i, out, n):
        self.log("download", i, n)
        for k, v in enumerate(self.held.get(i, [0.0] * n)):
            out[k] = v
        return 0

    def release(self, ids, n):
        self.log("release", ids[:n])
        for i in ids[:n]:
            self.sizes.pop(i, None)
        return 0

    def flush(self, words, n):
        self.log("flush", words[:n])
        return 0


@pytest.fixture
def rt():
    return RecordingRuntime()


@pytest.fixture
def graph(rt):
    return ComputeGraph(rt)


def bits(x):
    return struct.unpack("<i", struct.pack("<f", x))[0]


def test_constructor_rejects_null_and_new_graph_is_empty(graph):      # :21-30
    with pytest.raises(TypeError):
        ComputeGraph(None)
    assert graph.isEmpty()


def test_ensure_gpu_buffer_assigns_and_reuses(graph):                 # :34-52
    t = Tensor.from2D([[1, 2], [3, 4]])
    assert t.getGpuTag() is None
    buf = graph.ensureGpuBuffer(t)
    assert buf is t.getGpuTag() and (buf.rows, buf.cols) == (2, 2)
    assert graph.ensureGpuBuffer(t) is buf


def test_reupload_when_needs_upload(graph, rt):                       # :54-74
    t = Tensor.from2D([[1.0]])
    buf = graph.ensureGpuBuffer(t)
    buf.needsUpload = True
    t.data[0, 0] = 99.0
    graph.ensureGpuBuffer(t)
    assert not buf.needsUpload
    graph.flush()
    assert len(rt.uploads) == 2 and rt.uploads[1][1][0] == 99.0


def test_output_buffers(graph):                                       # :78-107
    buf = graph.newOutputBuffer(4, 8)
    assert buf.cpuStale and not buf.allocatedOnGpu and buf.floatCount() == 32
    a, b = graph.newOutputBuffer(1, 1), graph.newOutputBuffer(1, 1)
    assert b.id > a.id
    t = graph.createOutputTensor(graph.newOutputBuffer(3, 5))
    assert (t.rows, t.cols) == (3, 5) and isinstance(t.getGpuTag(), GpuBuffer)


def test_flush_on_empty_graph_is_noop_and_idempotent(graph, rt):      # :176-183,224-231
    for _ in range(3):
        graph.flush()
    assert not rt.allocCalls and not rt.uploads and not rt.flushCalls


def test_flush_allocates_uploads_executes_in_that_order(graph, rt):   # :185-210
    t = Tensor.from2D([[1, 2], [3, 4]])
    inp = graph.ensureGpuBuffer(t)
    out = graph.newOutputBuffer(2, 2)
    graph.recordUnary(op.OP_NEG, inp, out)
    graph.flush()
    assert len(rt.allocCalls) == 1 and list(rt.allocCalls[0][0]) == [inp.id, out.id]
    assert list(rt.allocCalls[0][1]) == [4, 4]
    assert len(rt.uploads) == 1 and rt.uploads[0][0] == inp.id
    assert len(rt.flushCalls) == 1
    assert list(rt.flushCalls[0][0]) == [op.OP_NEG, inp.id, out.id, 4]
    assert graph.isEmpty()                                            # :212-222


def test_second_flush_only_executes_new_ops(graph, rt):               # :233-253
    t = Tensor.from2D([[1]])
    inp = graph.ensureGpuBuffer(t)
    graph.recordUnary(op.OP_SQRT, inp, graph.newOutputBuffer(1, 1))
    graph.flush()
    graph.recordUnary(op.OP_NEG, inp, graph.newOutputBuffer(1, 1))
    graph.flush()
    assert len(rt.allocCalls) == 2 and len(rt.flushCalls) == 2 and len(rt.uploads) == 1


def test_a_runtime_that_clears_buffers_is_sent_no_zeros(rt):
    """A tensor nothing was written to is cleared by the runtime, before anything else of the flush is sent; one that was
    written to, with zeros or not, is sent, and so are all of them where the runtime has no such call."""
    events = []
    upload = rt.uploadBuffer

    def upload_logged(buf_id, data):
        events.append(("sent", buf_id))
        upload(buf_id, data)
    rt.uploadBuffer = upload_logged
    rt.zeroBuffers = lambda buffers: events.append(("cleared", list(buffers)))
    graph = ComputeGraph(rt)
    empty, touched, other = Tensor(2, 3), Tensor(2, 3), Tensor(4, 1)
    touched.data.fill(0.0)
    ids = [graph.ensureGpuBuffer(t).id for t in (touched, empty, other)]
    graph.flush()
    assert events == [("cleared", [(ids[1], 6), (ids[2], 4)]), ("sent", ids[0])]
    graph.flush()
    assert len(events) == 2

    plain = RecordingRuntime()
    g = ComputeGraph(plain)
    b = g.ensureGpuBuffer(Tensor(2, 3))
    g.flush()
    assert [u[0] for u in plain.uploads] == [b.id] and np.array_equal(plain.uploads[0][1], np.zeros(6, np.float32))


def test_ops_of_a_failed_flush_stay_recorded(graph, rt):
    """A refused stream has run nothing: its results stay stale, and the next attempt runs it instead of handing out what
    happens to be in their buffers."""
    b = graph.newOutputBuffer(2, 3)
    out = graph.createOutputTensor(b)
    graph.recordUnary(op.OP_EXP, graph.ensureGpuBuffer(Tensor(2, 3)), b)
    run, attempts = rt.flushOps, []

    def refuse_once(cmd, length):
        attempts.append(np.array(cmd[:length]).copy())
        if len(attempts) == 1:
            raise RuntimeError("workspace")
        run(cmd, length)
    rt.flushOps = refuse_once
    with pytest.raises(RuntimeError, match="workspace"):
        graph.materialize(out)
    assert b.cpuStale and not rt.downloads and not graph.isEmpty()
    graph.materialize(out)
    assert len(attempts) == 2 and np.array_equal(*attempts) and rt.downloads == [b.id] and graph.isEmpty()


def test_cmd_stream_grows_past_4096_ints(graph, rt):                  # :255-270
    a, b = graph.newOutputBuffer(2, 2), graph.newOutputBuffer(2, 2)
    for _ in range(1000):
        graph.recordBinary(op.OP_ADD, a, b, graph.newOutputBuffer(2, 2))
    graph.flush()
    assert len(rt.flushCalls) == 1 and rt.flushCalls[0][1] == 5000


def test_materialize_flushes_and_downloads_once(graph, rt):           # :274-333
    inp = graph.ensureGpuBuffer(Tensor.from2D([[2.0, 4.0]]))
    out = graph.newOutputBuffer(1, 2)
    graph.recordUnary(op.OP_SQRT, inp, out)
    result = graph.createOutputTensor(out)
    rt.downloadResult = [1.414, 2.0]
    graph.materialize(result)
    assert len(rt.flushCalls) == 1 and rt.downloads == [out.id]
    assert abs(result.data[0, 0] - 1.414) < 1e-3 and not out.cpuStale
    graph.materialize(result)
    assert len(rt.downloads) == 1
    graph.materialize(Tensor(2, 2))                                   # no GPU tag: no-op
    assert len(rt.downloads) == 1


def test_release_all_releases_resets_and_restarts_ids(graph, rt):     # :337-359,477-486
    t = Tensor.from2D([[1, 2]])
    graph.ensureGpuBuffer(t)
    graph.recordUnary(op.OP_NEG, graph.ensureGpuBuffer(t), graph.newOutputBuffer(1, 2))
    graph.releaseAll()
    assert len(rt.releaseCalls) == 1 and graph.isEmpty() and t.getGpuTag() is None
    assert graph.ensureGpuBuffer(Tensor.from2D([[9]])).id == 0
    g2 = ComputeGraph(RecordingRuntime())
    g2.releaseAll()
    assert not g2.runtime.releaseCalls


def test_release_all_materializes_stale_tracked_tensor(graph, rt):    # :392-408
    t = Tensor.from2D([[1.0]])
    buf = graph.ensureGpuBuffer(t)
    graph.flush()
    buf.cpuStale = True
    rt.downloadResult = [42.0]
    graph.releaseAll()
    assert t.data[0, 0] == 42.0 and t.getGpuTag() is None and not buf.cpuStale


def test_all_42_opcodes_are_distinct():                               # :362-390
    codes = list(op.REFERENCE_OPCODES.values())
    assert len(codes) == 42 and len(set(codes)) == 42 and sorted(codes) == list(range(1, 43))


def test_adamw_encodes_thirteen_ints(graph, rt):                      # :424-450
    w, g, mt, vt = (graph.newOutputBuffer(1, 4) for _ in range(4))
    graph.recordAdamWUpdate(w, g, mt, vt, 1e-3, 0.9, 0.999, 1e-8, 0.01, 0.9, 0.999, 4)
    graph.flush()
    stream, length = rt.flushCalls[0]
    assert length == 13
    assert list(stream) == [op.OP_ADAMW_UPDATE, w.id, g.id, mt.id, vt.id, bits(1e-3), bits(0.9), bits(0.999),
                            bits(1e-8), bits(0.01), bits(0.9), bits(0.999), 4]


def test_flush_marks_buffers_allocated_and_alloc_without_ops(graph, rt):   # :454-486
    t = Tensor.from2D([[1.0]])
    inp = graph.ensureGpuBuffer(t)
    out = graph.newOutputBuffer(1, 1)
    out_t = graph.createOutputTensor(out)
    assert not inp.allocatedOnGpu and not out.allocatedOnGpu
    graph.recordUnary(op.OP_NEG, inp, out)
    graph.flush()
    assert inp.allocatedOnGpu and out.allocatedOnGpu
    g2 = ComputeGraph(RecordingRuntime())
    g2.newOutputBuffer(2, 4)
    g2.flush()
    assert len(g2.runtime.allocCalls) == 1 and not g2.runtime.flushCalls
    del out_t


def test_orphaned_buffers_are_released_on_flush(graph, rt):           # :488-527
    t = Tensor.from2D([[1.0]])
    old = graph.ensureGpuBuffer(t)
    graph.flush()
    t.setGpuTag(graph.newOutputBuffer(1, 1))
    graph.flush()
    assert old.id in list(rt.releaseCalls[-1][0])
    t2 = Tensor.from2D([[2.0]])
    b2 = graph.ensureGpuBuffer(t2)
    graph.flush()
    t2.setGpuTag(None)
    n = len(rt.releaseCalls)
    graph.flush()
    assert len(rt.releaseCalls) == n + 1 and b2.id in list(rt.releaseCalls[-1][0])
    # a tensor that was garbage collected orphans its buffer too (WeakReference semantics)
    t3 = Tensor.from2D([[3.0]])
    b3 = graph.ensureGpuBuffer(t3).id
    graph.flush()
    del t3
    gc.collect()
    graph.flush()
    assert b3 in list(rt.releaseCalls[-1][0])


# ── HipBackend on top of the recording runtime: op -> stream mapping ─────────

def test_backend_records_reference_encodings(rt):
    be = HipBackend(rt)
    Tensor.setBackend(be)
    a, b = Tensor.from2D([[1, 2, 3], [4, 5, 6]]), Tensor.from2D([[7, 8], [9, 10], [11, 12]])
    c = be.matmul(a, b)
    d = c.multiplyScalar(0.5).addRowVector(Tensor.from2D([[1, 1]]))
    d.clamp(-1.0, 1.0)
    be.graph.flush()
    s = list(rt.flushCalls[0][0])
    ga, gb, gc_ = a.getGpuTag().id, b.getGpuTag().id, c.getGpuTag().id
    assert s[:7] == [op.OP_MATMUL, ga, gb, gc_, 2, 2, 3]              # [op,a,b,out,m,n,k]
    assert s[7] == op.OP_MULTIPLY_SCALAR and s[10] == bits(0.5) and s[11] == 4
    assert s[12] == op.OP_ADD_ROW_VECTOR and s[16:18] == [2, 2]
    assert s[18] == op.OP_CLAMP and s[21:24] == [bits(-1.0), bits(1.0), 4]


def test_backend_in_place_rebinds_to_new_buffer_and_releases_old(rt):  # MetalBackend.java:400-411
    be = HipBackend(rt)
    Tensor.setBackend(be)
    a, b = Tensor.from2D([[1.0, 2.0]]), Tensor.from2D([[3.0, 4.0]])
    be.graph.ensureGpuBuffer(a)
    old = a.getGpuTag().id
    a.addInPlace(b)
    assert a.getGpuTag().id != old and a.getGpuTag().cpuStale
    be.graph.flush()
    be.graph.flush()
    assert any(old in list(ids) for ids, _ in rt.releaseCalls)


def test_backend_shape_errors_before_recording(rt):                   # MetalBackendTest.java:80-86,271-276,315-323,364-372
    be = HipBackend(rt)
    Tensor.setBackend(be)
    with pytest.raises(ValueError, match="Shape mismatch"):
        be.matmul(Tensor(3, 4), Tensor(5, 2))
    with pytest.raises(ValueError, match="Shape mismatch"):
        be.softmaxBackward(Tensor(2, 3), Tensor(3, 2))
    with pytest.raises(ValueError, match="layerNormBackward: std"):
        be.layerNormBackward(Tensor(4, 8), Tensor(4, 8), Tensor(4, 2), 8)
    with pytest.raises(ValueError, match="targets length"):
        be.crossEntropyGradient(Tensor(4, 8), [0, 1, 2])
    assert be.graph.isEmpty()


def test_what_32_bit_words_cannot_count_is_refused(rt):
    class Clearing(RecordingRuntime):
        def zeroBuffers(self, zeros): pass

    runtime = Clearing()
    backend = HipBackend(runtime)
    big = Tensor(50000, 50000)                    # (its zeros are never made on the host)
    for call in (lambda: backend.add(big, big), lambda: backend.matmul(Tensor(70000, 1), Tensor(1, 70000)),
                 lambda: backend.transpose(Tensor(0, 1 << 31))):
        with pytest.raises(OverflowError):
            call()
    out = backend.add(Tensor(2, 2), Tensor(2, 2))
    backend.graph.flush()                         # what follows is recorded as ever
    assert all((sizes <= 70000).all() for _, sizes, _ in runtime.allocCalls) and len(runtime.flushCalls) == 1
    assert out.getGpuTag().allocatedOnGpu


def test_int_targets_travel_as_float_column(rt):                      # MetalBackend.java:43-54,531-539
    be = HipBackend(rt)
    Tensor.setBackend(be)
    be.crossEntropyGradient(Tensor(3, 5), [4, 0, 2])
    be.graph.flush()
    cols = [d for _, d in rt.uploads if d.size == 3]
    assert len(cols) == 1 and list(cols[0]) == [4.0, 0.0, 2.0]
    s = list(rt.flushCalls[0][0])
    assert s[0] == op.OP_CROSS_ENTROPY_GRADIENT and s[4:6] == [3, 5]


def test_tensors_graphs_and_copies_outlive_one_another():
    """A tensor tells every graph that tracks it when it goes, and a graph that is gone is told nothing; host tensors copy."""
    import copy
    import pickle
    first, second = RecordingRuntime(), RecordingRuntime()
    g1, g2 = ComputeGraph(first), ComputeGraph(second)
    t = Tensor.from2D([[1.0, 2.0]])
    buf = g1.ensureGpuBuffer(t).id
    assert g2.ensureGpuBuffer(t).id == buf and t.getGpuTag().graph is g2
    kept = g1.createOutputTensor(g1.newOutputBuffer(2, 2))
    g1.flush(), g2.flush()
    del t
    g1.flush(), g2.flush()
    assert [list(r.releaseCalls[-1][0]) for r in (first, second)] == [[buf], [buf]]
    del g1
    gc.collect()
    kept.setGpuTag(None)
    del kept

    # a buffer bound back to its tensor before the flush stays; one bound to another tensor belongs to that one
    a, b = Tensor.from2D([[1.0]]), Tensor.from2D([[2.0]])
    old = g2.ensureGpuBuffer(a)
    g2.flush()
    a.setGpuTag(None)
    a.setGpuTag(old)
    n = len(second.releaseCalls)
    g2.flush()
    assert len(second.releaseCalls) == n
    g2.bindTensorToBuffer(b, old)
    del a
    g2.flush()
    assert len(second.releaseCalls) == n
    del b
    g2.flush()
    assert list(second.releaseCalls[-1][0]) == [old.id]

    host = Tensor.from2D([[1.0, 2.0], [3.0, 4.0]])
    host.note = "kept"
    for c in (copy.copy(host), copy.deepcopy(host), pickle.loads(pickle.dumps(host))):
        assert (c.rows, c.cols, c.note) == (2, 2, "kept") and np.array_equal(c.data, host.data)
    assert copy.copy(host).data is host.data and copy.deepcopy(host).data is not host.data


@pytest.mark.parametrize("call", ["allocBuffers", "uploadBuffer", "flushOps", "releaseBuffers", "zeroBuffers"])
def test_a_runtime_may_flush_from_inside_a_call(call):
    """A runtime in Python that reads a tensor (and so flushes) while it is handed things: each thing is handed over, and nothing twice
    beside what the inner flush was handed again."""
    class Clearing(RecordingRuntime):
        def __init__(self):
            super().__init__()
            self.zeros = []

        def zeroBuffers(self, buffers):
            self.zeros.append(list(buffers))

    rt = Clearing()
    backend, depth = HipBackend(rt), [0]
    plain = getattr(rt, call)

    def again(*args):
        plain(*args)
        if depth[0] < 2:
            depth[0] += 1
            for k in range(20):                                        # (more of everything than the outer call holds)
                backend.add(Tensor.from2D([[1.0 + k]]), Tensor(1, 1))
            backend.graph.flush()
    setattr(rt, call, again)
    for round in range(3):
        kept = [backend.add(Tensor.from2D([[1.0, float(k)]]), Tensor(1, 2)) for k in range(30)]
        backend.graph.flush()
    assert backend.graph.isEmpty() and all(t.getGpuTag().allocatedOnGpu for t in kept)
    backend.releaseResources()


@pytest.mark.parametrize("fails", [False, True])
def test_a_read_releases_what_the_flush_in_front_of_it_has_orphaned(fails):
    """Behind the flush and in front of the download; and all the same where the download cannot be made."""
    lib = NativeLibrary()
    backend = HipBackend(lib.graph().runtime)
    a = Tensor.from2D([[1.0, 2.0]])
    for _ in range(2):
        dropped = backend.neg(a)
        kept = backend.exp(dropped)
        gone = dropped.getGpuTag().id
        del dropped
        if fails:
            kept._data = np.zeros((3, 3), np.float32)
            with pytest.raises(ValueError, match="Size mismatch"):
                backend.materializeTensor(kept)
        else:
            backend.materializeTensor(kept)
        names = [c[0] for c in lib.calls]
        assert names[-3:] == (["upload", "flush", "release"] if fails else ["flush", "release", "download"])
        assert gone in lib.calls[-1 if fails else -2][1] and gone not in lib.sizes and kept.getGpuTag().id in lib.sizes


def test_values_that_cannot_be_sent_are_the_flushs_to_report():
    """A large tensor's values are sent when it is first used.  One that cannot be sent then is recorded all the same, as a small one
    is, and leaves no buffer of its size to the next one; the flush says what is wrong, and sends it once that is over."""
    lib = NativeLibrary()
    graph = lib.graph()
    lib.fail_upload = True
    first = Tensor.from2D(np.ones((512, 512), np.float32))
    buf = graph.ensureGpuBuffer(first)
    assert not lib.sizes and not buf.allocatedOnGpu
    with pytest.raises(RuntimeError, match="the library says so"):
        graph.flush()
    lib.fail_upload = False
    second = Tensor.from2D(np.full((1024, 512), 2.0, np.float32))
    other = graph.ensureGpuBuffer(second)
    graph._emit(op.OP_NEG, buf.id, other.id, 512 * 512)
    graph.flush()
    assert lib.sizes == {buf.id: 512 * 512, other.id: 1024 * 512} and lib.held[other.id][-1] == 2.0 and lib.held[buf.id][-1] == 1.0


BLOCKING = """
#include <stdint.h>
#include <unistd.h>
volatile int block, inside, go, late, together;
static int active;
static int enter(int which) {
    if (__sync_fetch_and_add(&active, 1)) together = 1;
    if (block == which) {
        inside = 1;
        for (int i = 0; i < 50000 && !go; i++) usleep(100);
        if (!go) late = 1;
    } else usleep(block ? 0 : 20);
    __sync_fetch_and_sub(&active, 1);
    return 0;
}
int alloc(const int32_t *ids, const int32_t *sizes, int32_t n) { return enter(1); }
int upload(int32_t id, const float *v, int64_t n) { return enter(2); }
int flush(const int32_t *words, int32_t n) { return enter(3); }
int release(const int32_t *ids, int32_t n) { return enter(4); }
int download(int32_t id, float *v, int64_t n) { return enter(5); }
const char *error(void) { return "none"; }
"""
CALLS = ("alloc", "upload", "flush", "release", "download", "error")


@pytest.fixture
def blocking(tmp_path):
    """A library in C: no call of it needs the interpreter, and one of them waits until it is let go (5 s at most)."""
    (tmp_path / "blocking.c").write_text(BLOCKING)
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", str(tmp_path / "blocking.so"), str(tmp_path / "blocking.c")], check=True)
    lib = C.CDLL(str(tmp_path / "blocking.so"))
    lib.value = {n: C.c_int.in_dll(lib, n) for n in ("block", "inside", "go", "late", "together")}

    class Runtime:
        nativeCalls = staticmethod(lambda: tuple(C.cast(getattr(lib, n), C.c_void_p).value for n in ("alloc", "upload", "download", "release", "flush", "error")))
        def zeroBuffers(self, buffers): raise AssertionError("not called where the library is")
        def hostArray(self, n): return np.empty(n, np.float32)
    lib.runtime = Runtime
    return lib


@pytest.mark.parametrize("call", range(1, 7), ids=(*CALLS[:5], "large upload"))
def test_other_threads_run_and_record_while_a_call_of_the_library_waits(blocking, call):
    state, backend = blocking.value, HipBackend(blocking.runtime())
    graph, a, b = backend.graph, Tensor.from2D([[1.0, 2.0]]), Tensor.from2D([[3.0, 4.0]])
    backend.add(a, b)                                                  # a result nobody keeps: the flush releases it
    kept = backend.multiply(a, b)
    large = Tensor.from2D(np.ones((512, 1024), np.float32))
    state["block"].value = min(call, 5) if call < 6 else 2
    worker = threading.Thread(target=lambda: kept.materialize() if call < 6 else graph.ensureGpuBuffer(large), daemon=True)
    Tensor.setBackend(backend)
    worker.start()
    until = time.monotonic() + 4
    while not state["inside"].value and time.monotonic() < until:
        time.sleep(0.001)
    more = backend.subtract(a, Tensor.from2D([[5.0, 6.0]]))            # recorded meanwhile: the next flush's
    state["go"].value = 1
    worker.join()
    assert state["inside"].value and not state["late"].value and not state["together"].value
    assert not graph.isEmpty() and not more.getGpuTag().allocatedOnGpu
    graph.flush()
    assert graph.isEmpty() and more.getGpuTag().allocatedOnGpu
    if call == 6:
        assert large.getGpuTag().allocatedOnGpu


def test_an_operand_may_get_another_buffer_while_the_other_ones_values_are_sent():
    """A host array of some other class runs code of its own when it is packed; here it takes the other operand's buffer away."""
    runtime = RecordingRuntime()
    backend = HipBackend(runtime)
    a, b = Tensor.from2D([[1.0, 2.0]]), Tensor(1, 2)

    class Taking:
        def astype(self, dtype, order):
            a.setGpuTag(None)
            gc.collect()
            [GpuBuffer(100 + k, 7, 7, False) for k in range(64)]       # (what may get the memory)
            return np.array([[3.0, 4.0]], np.float32)
    b._data = Taking()
    first = backend.graph.ensureGpuBuffer(a).id
    backend.graph.flush()                                              # (what waits to be made would hold it)
    out = backend.add(a, b)
    backend.graph.flush()
    words = [list(c[0]) for c in runtime.flushCalls]
    assert words == [[op.OP_ADD, first, b.getGpuTag().id, out.getGpuTag().id, 2]]


def test_the_librarys_calls_run_one_at_a_time(blocking):
    """It asks that of its callers; graphs of several threads keep to it."""
    def work(backend):
        for _ in range(30):
            x = Tensor.from2D(np.ones((512, 512), np.float32))
            y = backend.add(x, Tensor.from2D(np.ones((512, 512), np.float32)))
            backend.materializeTensor(y)
            del x, y
    threads = [threading.Thread(target=work, args=(HipBackend(blocking.runtime()),)) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not blocking.value["together"].value


class CountingGraph(ComputeGraph):
    """Every method an operation goes through, counted."""

    def __init__(self, runtime):
        super().__init__(runtime)
        self.seen = []


for _name in ("ensureGpuBuffer", "newOutputBuffer", "createOutputTensor", "bindTensorToBuffer", "tensorLetGo", "flush", *(n for n in dir(ComputeGraph) if n.startswith("record"))):
    def _counting(self, *args, _name=_name):
        self.seen.append(_name)
        return getattr(ComputeGraph, _name)(self, *args)
    setattr(CountingGraph, _name, _counting)


def _every_operation(be):
    """Each operation of the backend once, over operands of its own; what it hands back."""
    t = lambda r, c, first=1.0: Tensor.from2D(np.arange(first, first + r * c, dtype=np.float32).reshape(r, c))
    m, row, col, results = t(2, 3), t(1, 3), t(2, 1), []
    for name in ("add", "subtract", "multiply", "divide", "reluBackward", "geluBackward", "softmaxBackward"):
        results.append(getattr(be, name)(m, t(2, 3, 4.0)))
    for name in ("addInPlace", "subtractInPlace", "multiplyInPlace", "divideInPlace"):
        x = t(2, 3, 2.0)
        results += [getattr(be, name)(x, m), x]
    for name in ("sqrt", "neg", "exp", "log", "tanh", "sigmoid", "relu", "gelu", "transpose", "softmaxRows", "sumRows", "sumAlongRows", "meanAlongRows",
                 "varianceAlongRows", "maxAlongRows"):
        results.append(getattr(be, name)(m))
    for name in ("sqrtInPlace", "negInPlace", "expInPlace", "logInPlace", "reluInPlace", "geluInPlace", "tanhInPlace", "sigmoidInPlace"):
        x = t(2, 3, 3.0)
        results += [getattr(be, name)(x), x]
    for name in ("multiplyScalar", "addScalar", "divideScalar", "pow"):
        results.append(getattr(be, name)(m, 1.5))
    for name in ("multiplyScalarInPlace", "addScalarInPlace", "divideScalarInPlace"):
        x = t(2, 3, 5.0)
        results += [getattr(be, name)(x, 2.5), x]
    results += [be.addRowVector(m, row), be.multiplyBroadcastRows(m, row)]
    results += [getattr(be, name)(m, col) for name in ("addBroadcastCols", "subtractBroadcastCols", "divideBroadcastCols", "multiplyBroadcastCols")]
    results += [be.matmul(m, t(3, 4)), be.clamp(m, 0.0, 1.0), be.sum(m), be.sumAbs(m), be.crossEntropyLoss(m, [0, 1]), be.crossEntropyGradient(m, [2, 0])]
    w, mt, vt = t(2, 3), t(2, 3), t(2, 3)
    results += [be.adamWUpdate(w, m, mt, vt, 1e-3, 0.9, 0.99, 1e-8, 0.0, 1.0, 1.0), w, mt, vt, be.layerNormBackward(m, t(2, 3), col, 3)]
    for call, bad in ((be.add, (m, row)), (be.matmul, (m, m)), (be.addRowVector, (m, col)), (be.addBroadcastCols, (m, row)), (be.multiplyInPlace, (m, col))):
        with pytest.raises(ValueError) as e:
            call(*bad)
        results.append(str(e.value))
    be.graph.flush()
    return [r.getGpuTag().id if isinstance(r, Tensor) else r for r in results]


def _calls(runtime):
    return [[(list(a), list(b)) for a, b, _ in runtime.allocCalls], [(i, list(v)) for i, v in runtime.uploads], runtime.downloads,
            [list(c) for c, _ in runtime.flushCalls], [list(a) for a, _ in runtime.releaseCalls]]


class Forwarding:
    """An object that is no ComputeGraph and passes everything on to one."""

    def __init__(self, runtime): self.inner = ComputeGraph(runtime)
    def __getattr__(self, name): return getattr(self.inner, name)


@pytest.mark.parametrize("way", ["subclass", "instance", "class", "other object"])
def test_methods_of_a_graph_that_are_replaced_are_called(way, monkeypatch):
    """By a class derived from ComputeGraph, on one graph, on ComputeGraph itself, or by an object in its place: the operations go
    through the methods, and record and hand back what they do otherwise."""
    plain_rt, rt = RecordingRuntime(), RecordingRuntime()
    plain = HipBackend(plain_rt)
    Tensor.setBackend(plain)
    want = _every_operation(plain)
    be, seen = HipBackend(rt), []
    if way == "subclass":
        be.graph = CountingGraph(rt)
        seen = be.graph.seen
    elif way == "instance":
        record = be.graph.recordBinary
        be.graph.recordBinary = lambda *a: (seen.append("recordBinary"), record(*a))
    elif way == "class":
        record = ComputeGraph.recordBinary
        monkeypatch.setattr(ComputeGraph, "recordBinary", lambda self, *a: (seen.append("recordBinary"), record(self, *a))[1])
    else:
        be.graph = Forwarding(rt)
        seen.append("recordBinary")
    Tensor.setBackend(be)
    assert _every_operation(be) == want
    assert _calls(rt) == _calls(plain_rt)
    assert "recordBinary" in seen
    if way == "subclass":
        assert set(seen) == {n for n in dir(CountingGraph) if not n.startswith("_")} - {
            "recordScatterAddRows", "recordScatterAddRowsAtomic", "runtime", "isEmpty", "materialize", "releaseAll", "seen"}
    monkeypatch.undo()
    n = len(seen)
    if way == "class":
        be.add(Tensor(1, 1), Tensor(1, 1))
        assert len(seen) == n                                          # and the short way is back


@pytest.mark.parametrize("owner,names", [(HipGpuRuntime, ("allocBuffers", "uploadBuffer", "downloadBuffer", "releaseBuffers", "flushOps", "zeroBuffers")),
                                         (HipNative, ("nativeAllocBuffers", "nativeUploadBuffer", "nativeDownloadBuffer", "nativeReleaseBuffers", "nativeFlushOps"))])
def test_calls_of_the_runtime_that_are_replaced_are_called(owner, names, monkeypatch):
    """On the classes that pass them on to the library; a large tensor's values too, and back."""
    seen = []
    for name in names:
        if owner is HipNative:
            monkeypatch.setattr(owner, name, staticmethod(lambda *a, name=name: seen.append(name)))
        else:
            monkeypatch.setattr(owner, name, lambda self, *a, name=name: seen.append(name))
    be = HipBackend()
    out = be.add(be.add(Tensor.from2D(np.ones((512, 512), np.float32)), Tensor(512, 512)), Tensor(512, 512))
    be.graph.flush()
    be.materializeTensor(out)
    del out
    be.graph.flush()
    assert set(seen) == set(names)
    be.releaseResources()


def test_a_tensor_class_with_values_of_its_own_has_them_sent():
    class Doubled(Tensor):
        @property
        def data(self):
            return 2 * super().data
    rt = RecordingRuntime()
    be = HipBackend(rt)
    t = Doubled(1, 2)
    t._data = np.array([[1.0, 2.0]], np.float32)
    out = be.add(t, Tensor.from2D([[0.0, 0.0]]))
    be.graph.flush()
    assert [list(v) for _, v in rt.uploads] == [[2.0, 4.0], [0.0, 0.0]] and out.getGpuTag().allocatedOnGpu
    held = t.getGpuTag().id
    del t
    be.graph.flush()
    assert list(rt.releaseCalls[-1][0]) == [held]


class Matrix:
    """No Tensor, but all that a graph asks of one."""

    def __init__(self, rows, cols, values=None):
        self.rows, self.cols, self._gpu_tag, self._data = rows, cols, None, values

    @property
    def data(self):
        if self._data is None:
            self._data = np.zeros((self.rows, self.cols), np.float32)
        return self._data

    def setGpuTag(self, tag):
        old, self._gpu_tag = self._gpu_tag, tag
        if old is not None and old is not tag:
            old.graph.tensorLetGo(old)


def _host_tensor(values):
    t = Tensor(*values.shape)
    t._data = values
    return t


def test_objects_that_stand_in_for_a_tensor_are_taken():
    """An object with a tensor's attributes as operand, in place, read back, dropped and released: the calls that tensors make."""
    calls = []
    for make in (_host_tensor, lambda v: Matrix(*v.shape, v)):
        rt = RecordingRuntime()
        rt.downloadResult = [9.0, 8.0, 7.0, 6.0]
        be = HipBackend(rt)
        Tensor.setBackend(be)
        a, b = make(np.array([[1, 2], [3, 4]], np.float32)), make(np.array([[5, 6], [7, 8]], np.float64).T)
        blank = make(np.zeros((2, 2), np.float32)) if make is _host_tensor else Matrix(2, 2)
        dropped = be.add(a, b)
        be.multiplyInPlace(a, blank)
        be.materializeTensor(a)
        assert a._data.tolist() == [[9, 8], [7, 6]] and not a._gpu_tag.cpuStale
        out = be.matmul(b, a)
        b._gpu_tag.needsUpload = True
        be.addScalarInPlace(b, 1.0)
        be.reluInPlace(b)
        del dropped
        be.materializeTensor(out)
        held = blank._gpu_tag.id
        del blank
        be.graph.flush()
        assert list(rt.releaseCalls[-1][0]) == [held]
        be.subtract(a, out)
        be.releaseResources()
        assert a._gpu_tag is None and b._gpu_tag is None and b._data.tolist() == [[9, 8], [7, 6]]
        calls.append(_calls(rt))
    plain, other = calls
    assert other == plain
    graph = ComputeGraph(RecordingRuntime())
    with pytest.raises(TypeError):
        graph.materialize(np.zeros((1, 1)))
    m, t = Matrix(1, 1), Tensor(1, 1)
    buf = graph.ensureGpuBuffer(m)                                     # from one kind to the other and back
    graph.bindTensorToBuffer(t, buf)
    m.setGpuTag(None)
    graph.flush()
    assert not graph.runtime.releaseCalls
    graph.bindTensorToBuffer(m, buf)
    t.setGpuTag(None)
    graph.flush()
    assert not graph.runtime.releaseCalls
    gone = weakref.ref(graph)
    del graph, buf
    m.setGpuTag(None)
    gc.collect()
    assert gone() is None


def test_sizes_and_flags_take_what_counts():
    """numpy's integers and truth values, as attributes of a class in Python do."""
    t, b = Tensor(2, 3), GpuBuffer(1, 2, 3, False)
    for o in (t, b):
        for name, value in (("rows", np.int64(4)), ("cols", np.int32(5)), ("rows", True), ("cols", 6)):
            setattr(o, name, value)
            assert getattr(o, name) == value and type(getattr(o, name)) is int
        for wrong in ("a", None):
            with pytest.raises((TypeError, ValueError)):
                o.rows = wrong
        assert (o.rows, o.cols) == (1, 6)
    for name in ("needsUpload", "cpuStale", "allocatedOnGpu"):
        for value in (np.bool_(True), 0, 1, False):
            setattr(b, name, value)
            assert getattr(b, name) is bool(value)
    b.id = np.int64(7)
    assert b.id == 7 and b.floatCount() == 6


def test_a_tensor_class_with_a_set_gpu_tag_of_its_own_has_it_called():
    class Watching(Tensor):
        def setGpuTag(self, tag):
            self.__dict__.setdefault("tags", []).append(tag)
            super().setGpuTag(tag)
    be = HipBackend(RecordingRuntime())
    t = Watching(1, 2)
    t.data[:] = 1.0
    be.negInPlace(t)
    be.releaseResources()
    assert [type(x) for x in t.tags] == [GpuBuffer, GpuBuffer, type(None)] and t.tags[0] is not t.tags[1]


@pytest.mark.parametrize("holder", ["graph", "runtime", "tensor"])
def test_cycles_through_tensors_are_collected(holder):
    """A graph, a runtime or a tensor that keeps a tensor of the graph's (or itself): all of it goes when the program lets go."""
    runtime = RecordingRuntime()
    graph = ComputeGraph(runtime)
    t = Tensor.from2D([[1.0, 2.0]])
    graph.ensureGpuBuffer(t)
    graph.flush()
    out = graph.createOutputTensor(graph.newOutputBuffer(2, 2))         # (its buffer is still to be made)
    {"graph": graph, "runtime": runtime, "tensor": t}[holder].kept = [t, out]
    gone = [weakref.ref(o) for o in (graph, t, out)]
    del graph, runtime, t, out
    gc.collect()
    assert [r() for r in gone] == [None] * 3


@pytest.mark.parametrize("make", [_host_tensor, lambda v: Matrix(*v.shape, v)])
def test_results_reach_a_tensor_whose_host_array_cannot_be_written(graph, rt, make):
    """A view of bytes, of a file mapped to be read: the tensor gets an array of its own, and what it was made from stays as it is."""
    raw = np.array([1.0, 2.0], np.float32).tobytes()
    t = make(np.frombuffer(raw, np.float32).reshape(1, 2))
    buf = graph.ensureGpuBuffer(t)
    graph.flush()
    rt.downloadResult = [5.0, 6.0]
    for release in (lambda: graph.materialize(t), graph.releaseAll):
        buf.cpuStale = True
        release()
        assert t.data.tolist() == [[5.0, 6.0]] and t.data.flags.writeable
        assert raw == np.array([1.0, 2.0], np.float32).tobytes()
        rt.downloadResult = [5.0, 6.0]


def test_a_tensor_saved_as_its_attributes_loads():
    """As tensors were pickled while all they held was in their dictionary, and as a derived class may save itself."""
    state = {"_gpu_tag": None, "_data": np.array([[1.0, 2.0]], np.float32), "rows": 1, "cols": 2, "note": "kept"}
    t = Tensor.__new__(Tensor)
    t.__setstate__(state)
    assert (t.rows, t.cols, t.note, t.getGpuTag()) == (1, 2, "kept", None) and t.numpy().tolist() == [[1.0, 2.0]]


def test_values_of_other_layouts_travel_as_fp32_rows(graph, rt):
    """Host arrays that are not contiguous fp32 are packed on the way out, filled on the way back; a size that does not fit is refused."""
    t = Tensor(2, 3)
    t.data = np.arange(6, dtype=np.float64).reshape(3, 2).T
    buf = graph.ensureGpuBuffer(t)
    graph.flush()
    assert list(rt.uploads[0][1]) == [0, 2, 4, 1, 3, 5] and rt.uploads[0][1].dtype == np.float32
    buf.cpuStale = True
    rt.downloadResult = [5, 4, 3, 2, 1, 0]
    graph.materialize(t)
    assert t.data.dtype == np.float64 and t.data.tolist() == [[5, 4, 3], [2, 1, 0]]
    small = Tensor(1, 2)
    small.data.fill(1)
    small.setGpuTag(graph.newOutputBuffer(3, 3))
    with pytest.raises(ValueError, match="Size mismatch"):
        graph.materialize(small)
    with pytest.raises(TypeError):
        graph.ensureGpuBuffer(np.zeros((2, 2)))
