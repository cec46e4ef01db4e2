"""Consecutive element-wise operations run as one launch: the same bits as each of them by itself, whatever they read and
write in common."""
import numpy as np
import pytest

from deepj_amd import HipNative, opcodes as op
from deepj_amd.fused import DeviceBuffers, Stream

pytestmark = pytest.mark.gpu

BINARY = [op.OP_ADD, op.OP_SUBTRACT, op.OP_MULTIPLY, op.OP_DIVIDE, op.OP_RELU_BACKWARD, op.OP_GELU_BACKWARD]
UNARY = [op.OP_SQRT, op.OP_NEG, op.OP_EXP, op.OP_LOG, op.OP_TANH, op.OP_SIGMOID, op.OP_RELU, op.OP_GELU]
SCALAR = [op.OP_MULTIPLY_SCALAR, op.OP_ADD_SCALAR, op.OP_DIVIDE_SCALAR, op.OP_POW]
ROWS = [op.OP_ADD_ROW_VECTOR, op.OP_MULTIPLY_BROADCAST_ROWS]
COLS = [op.OP_ADD_BROADCAST_COLS, op.OP_SUBTRACT_BROADCAST_COLS, op.OP_DIVIDE_BROADCAST_COLS, op.OP_MULTIPLY_BROADCAST_COLS]


def _bits(x):
    return int(np.float32(x).view(np.int32))


def _program(rng, rows, cols, length):
    """(ops, buffers): words with buffer indexes; 0 .. 5 hold rows x cols values, 6, 7 a row, 8, 9 a column, 10, 11 square operands."""
    n, ops = rows * cols, []
    full = lambda: int(rng.integers(0, 6))
    for _ in range(length):
        kind = int(rng.integers(0, 8))
        a, b, out = full(), full(), full()
        if kind <= 1:
            ops.append([int(rng.choice(BINARY)), a, b, out, n])
        elif kind == 2:
            ops.append([int(rng.choice(UNARY)), a, out, n])
        elif kind == 3:
            ops.append([int(rng.choice(SCALAR)), a, out, _bits(rng.uniform(0.5, 1.5)), n])
        elif kind == 4:
            ops.append([op.OP_CLAMP, a, out, _bits(-1.5), _bits(2.0), n])
        elif kind == 5:
            ops.append([int(rng.choice(ROWS)), a, int(rng.integers(6, 8)), out, rows, cols])
        elif kind == 6:
            ops.append([int(rng.choice(COLS)), a, int(rng.integers(8, 10)), out, rows, cols])
        else:
            ops.append([op.OP_MATMUL, int(rng.integers(10, 12)), a, out, rows, cols, rows] if rng.random() < 0.7 and out != a
                       else [op.OP_SUM_ALONG_ROWS, a, int(rng.integers(8, 10)), rows, cols])
    return ops


SLOTS = {5: (1, 2, 3), 4: (1, 2), 6: (1, 2, 3), 7: (1, 2, 3)}


def _ids(word, ids):
    code = word[0]
    if code in UNARY or code in SCALAR or code in (op.OP_CLAMP, op.OP_SUM_ALONG_ROWS):
        at = (1, 2)
    else:
        at = (1, 2, 3)
    return [ids[w] if i in at else w for i, w in enumerate(word)]


@pytest.mark.parametrize("rows,cols", [(1, 1), (1, 3), (5, 1), (3, 5), (7, 64), (33, 130), (64, 257), (300, 41)])
def test_a_chain_has_the_bits_of_its_operations(rows, cols):
    rng = np.random.default_rng(rows * 1000 + cols)
    for trial in range(40):
        ops = _program(rng, rows, cols, int(rng.integers(2, 24)))
        shapes = [rows * cols] * 6 + [cols] * 2 + [rows] * 2 + [rows * rows] * 2
        values = [(rng.standard_normal(s) * (1.0 if i < 10 else rows ** -0.5)).astype(np.float32) for i, s in enumerate(shapes)]
        if trial % 8 == 0:
            values[0][0], values[1][-1], values[2][0] = np.inf, np.nan, -0.0
        results = []
        for together in (True, False):
            dev = DeviceBuffers()
            try:
                ids = [dev.upload(v) for v in values]
                if together:
                    s = Stream()
                    for o in ops:
                        s.emit(*_ids(o, ids))
                    s.run()
                else:
                    for o in ops:
                        Stream().emit(*_ids(o, ids)).run()
                results.append([dev.download(b, (n,)) for b, n in zip(ids, shapes)])
            finally:
                dev.release_all()
        for k, (x, y) in enumerate(zip(*results)):
            same = (x.view(np.uint32) == y.view(np.uint32)) | (np.isnan(x) & np.isnan(y))
            assert same.all(), (trial, k, ops)


@pytest.mark.parametrize("rows,cols,least", [(255, 513, 3), (257, 511, 2), (1021, 1027, 2), (1025, 1031, 4), (2051, 4111, 4)])
def test_the_operations_that_make_a_chain(rows, cols, least):
    """From how many operations on they run as one launch, at sizes on either side of each rule (2^17 and 2^20 values) and past what
    one pass of a launch covers (2^23), none a multiple of four, vectors of both kinds among the operands: one launch, and the bits
    of the operations one by one."""
    rng, n = np.random.default_rng(rows), rows * cols
    a, b, row, col = (rng.standard_normal(s).astype(np.float32) for s in (n, n, cols, rows))
    dev = DeviceBuffers()
    try:
        A, B, R, C = (dev.upload(v) for v in (a, b, row, col))
        outs = [dev.alloc(n) for _ in range(4)]
        words = [[op.OP_MULTIPLY_BROADCAST_COLS, A, C, outs[0], rows, cols], [op.OP_ADD_ROW_VECTOR, outs[0], R, outs[1], rows, cols],
                 [op.OP_SIGMOID, outs[1], outs[2], n], [op.OP_SUBTRACT, outs[2], B, outs[3], n]]
        for length in (2, 3, 4):
            stream = Stream()
            for w in words[:length]:
                stream.emit(*w)
                Stream().emit(*w).run()
            want = [dev.download(o, (n,)).copy() for o in outs[:length]]
            for o in outs:
                Stream().fill(o, 0, n).run()
            stream.run()
            for o, x in zip(outs, want):
                assert np.array_equal(dev.download(o, (n,)).view(np.uint32), x.view(np.uint32))
            launches = [int(c) for c in HipNative.profileOps(stream.array(), 1, detail=True)[2]]
            assert launches == ([1] + [0] * (length - 1) if length >= least else [1] * length), (length, launches)
    finally:
        dev.release_all()


def test_values_that_need_a_ninth_slot_run_in_shorter_chains():
    """Six operands and three results needed to the end are more than a chain holds: the same bits all the same."""
    rng, n = np.random.default_rng(1), 1000
    dev = DeviceBuffers()
    try:
        e = [dev.upload(rng.standard_normal(n).astype(np.float32)) for _ in range(6)]
        r = [dev.alloc(n) for _ in range(8)]
        words = [[op.OP_ADD, e[0], e[1], r[0], n], [op.OP_SUBTRACT, e[2], e[3], r[1], n], [op.OP_MULTIPLY, e[4], e[5], r[2], n], [op.OP_ADD, e[0], r[0], r[3], n],
                 [op.OP_MULTIPLY, e[1], e[2], r[4], n], [op.OP_SUBTRACT, r[3], r[1], r[5], n], [op.OP_ADD, e[3], e[4], r[6], n], [op.OP_DIVIDE, r[2], e[5], r[7], n]]
        for w in words:
            Stream().emit(*w).run()
        want = [dev.download(o, (n,)).copy() for o in r]
        stream = Stream()
        for w in words:
            stream.emit(*w)
        for o in r:
            Stream().fill(o, 0, n).run()
        stream.run()
        assert all(np.array_equal(dev.download(o, (n,)), x) for o, x in zip(r, want))
        launches = [int(c) for c in HipNative.profileOps(stream.array(), 1, detail=True)[2]]
        assert launches[0] == 1 and launches[1] == 1 and sum(launches) < len(words), launches
    finally:
        dev.release_all()


def test_transposes_of_any_shape_in_one_launch():
    """Eight that depend on nothing, of different rows and columns (one tile, a tile's edge on either side, rows, columns), between
    operations that they go past: all in the first one's launch."""
    rng = np.random.default_rng(2)
    shapes = [(1, 70), (70, 1), (32, 32), (33, 31), (5, 257), (300, 40), (64, 1003), (31, 97)]
    dev = DeviceBuffers()
    try:
        values = [rng.standard_normal(s).astype(np.float32) for s in shapes]
        ins, outs = [dev.upload(v) for v in values], [dev.alloc(v.size) for v in values]
        x = dev.upload(rng.standard_normal((20, 30)).astype(np.float32))
        stream = Stream()
        for (rows, cols), i, o in zip(shapes, ins, outs):
            stream.emit(op.OP_TRANSPOSE, i, o, rows, cols).emit(op.OP_EXP, x, x, 600)
        stream.run()
        for v, o in zip(values, outs):
            assert np.array_equal(dev.download(o, v.T.shape), v.T)
        launches = [int(c) for c in HipNative.profileOps(stream.array(), 1, detail=True)[2]]
        assert launches == [1, 1] + [0, 1] * 7, launches
    finally:
        dev.release_all()


def test_a_product_between_two_operations_that_depends_on_one_of_them_stays_there():
    """x = a + b; y = m . x; z = y * x: the product reads a result in front of it, and overwrites an operand behind it."""
    rng = np.random.default_rng(0)
    a, b, m = (rng.standard_normal((32, 32)).astype(np.float32) for _ in range(3))
    dev = DeviceBuffers()
    try:
        A, B, M, X, Z = dev.upload(a), dev.upload(b), dev.upload(m), dev.alloc(1024), dev.alloc(1024)
        s = Stream().emit(op.OP_ADD, A, B, X, 1024).matmul(M, X, A, 32, 32, 32).emit(op.OP_MULTIPLY, A, X, Z, 1024).emit(op.OP_NEG, Z, B, 1024)
        s.run()
        got = dev.download(B, (32, 32))
    finally:
        dev.release_all()
    x = (a + b).astype(np.float64)
    exp = -(m.astype(np.float64) @ x) * x
    bound = 2 * 33 * 2.0 ** -24 * (np.abs(m).astype(np.float64) @ np.abs(x)) * np.abs(x)
    assert np.all(np.abs(got - exp) <= bound)


@pytest.mark.parametrize("n", [1, 5, 32, 33, 70, 200])
def test_transposes_that_run_ahead_change_no_bit(n):
    """Streams of transposes, products, sums and reductions over few square buffers, so that most transposes depend on what stands
    in front of them: the bits of the operations one by one."""
    rng = np.random.default_rng(n)
    dev = DeviceBuffers()
    try:
        start = (rng.standard_normal((8, n, n)) * n ** -0.5).astype(np.float32)
        ids = [dev.alloc(n * n) for _ in range(8)]
        rows = [dev.alloc(n) for _ in range(2)]

        def run(ops, together):
            for i, a in zip(ids, start):
                dev.write(i, a)
            for r in rows:
                dev.write(r, np.zeros(n, np.float32))
            if together:
                s = Stream()
                for o in ops:
                    s.emit(*o)
                s.run()
            else:
                for o in ops:
                    Stream().emit(*o).run()
            return [dev.download(i, (n, n)).copy() for i in ids] + [dev.download(r, (n,)).copy() for r in rows]
        for length in (2, 3, 9, 40, 80):
            ops = []
            for _ in range(length):
                a, b, out = (int(x) for x in rng.choice(ids, 3, replace=False))
                kind = int(rng.integers(0, 10))
                if kind < 5:
                    ops.append([op.OP_TRANSPOSE, a, out, n, n])
                elif kind < 7:
                    ops.append([op.OP_MATMUL, a, b, out, n, n, n])
                elif kind == 7:
                    ops.append([op.OP_SUBTRACT, a, b, out, n * n])
                elif kind == 8:
                    ops.append([op.OP_SUM_ROWS, a, int(rng.choice(rows)), n, n])
                else:
                    ops.append([op.OP_ADD_ROW_VECTOR, a, int(rng.choice(rows)), out, n, n] if rng.random() < 0.8 else [op.OP_EXP, a, a, n * n])
            for got, want in zip(run(ops, True), run(ops, False)):
                assert np.array_equal(got, want, equal_nan=True)
    finally:
        dev.release_all()
