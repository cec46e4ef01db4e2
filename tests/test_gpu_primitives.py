"""GPU-vs-CPU differential tests of the 42 primitive opcodes through HipBackend ->
ComputeGraph -> C ABI -> HIP kernels, against the CPU oracle on the same seeded inputs.
Shapes, seeds and tolerances follow the reference's own GPU test
src/test/java/io/github/kirstenali/deepj/tensor/metal/MetalBackendTest.java (cited per test);
where that test loosened a tolerance "because fast-math exp", this one does not have to."""
import numpy as np
import pytest

from deepj_amd import HipNative, Tensor
from deepj_amd import opcodes as op
from deepj_amd.fused import DeviceBuffers, Stream
from oracle import cpu_ref as ref
from gpu_util import assert_close, backend, rnd, tensor

pytestmark = pytest.mark.gpu


def test_native_is_available():                                       # :41-44
    assert HipNative.available()


def test_small_matmul_matches_expected_values():                      # :46-68
    with backend() as be:
        c = be.matmul(tensor([[1, 2, 3], [4, 5, 6]]), tensor([[7, 8], [9, 10], [11, 12]]))
        assert (c.rows, c.cols) == (2, 2)
        assert_close([[58, 64], [139, 154]], c, atol=1e-6, rtol=0)


@pytest.mark.parametrize("m,k,n", [(128, 192, 64), (1, 2048, 513), (65, 33, 127), (200, 513, 70), (3, 1, 5),
                                   (1100, 257, 2050), (1536, 64, 1537)])       # large enough for the 128 x 128 tile, ragged
def test_matmul_matches_cpu(m, k, n):                                 # :70-78 (+ ragged shapes)
    a, b = rnd(m, k, 1), rnd(k, n, 2)
    with backend() as be:
        assert_close(ref.matmul(a, b), be.matmul(tensor(a), tensor(b)), 1e-4, 1e-4, f"matmul {m}x{k}x{n}")


@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (1, 33, 7), (31, 32, 8), (33, 65, 31), (32, 64, 256), (64, 96, 257), (40, 300, 515),
                                   (97, 2000, 40), (256, 1003, 129), (320, 2752, 36), (500, 2700, 260), (1030, 1100, 130), (900, 4100, 68),
                                   (2100, 1000, 37), (1030, 2756, 1), (1024, 2752, 31), (1090, 2760, 36), (1000, 7000, 133),
                                   (3001, 2047, 65), (4100, 2052, 260)])
def test_matmul_tiles_and_remainders(m, n, k):
    """Every tile of the dispatch with rows, columns and K that do not fill it, and K below, at and past a stage of its
    loop.  Bound: a sum of k products in any order is off by at most k * 2^-24 * sum |a||b| (first order; the 2 covers the
    second)."""
    rng = np.random.default_rng(m * n + k)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    with backend() as be:
        got = be.matmul(tensor(a), tensor(b)).numpy().astype(np.float64)
    bound = 2 * k * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64))
    assert np.all(np.abs(got - a.astype(np.float64) @ b.astype(np.float64)) <= bound)


@pytest.mark.parametrize("m,n,k", [(1, 1, 257), (2, 17, 264), (16, 16, 260), (17, 33, 272), (33, 47, 511), (256, 192, 1003), (15, 4097, 271),
                                   (512, 256, 304), (513, 256, 304), (4, 2752, 1024), (100, 300, 4001)])
def test_matmul_of_small_outputs_over_a_long_k(m, n, k):
    """Tiles of 16 x 16 that sixteen wavefronts share the K of: an element past a tile, a stage (16) and a round of them (256), the
    most tiles there are and one row more, under the same bound; a NaN stays in its row."""
    rng = np.random.default_rng(m + n * k)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    exact = a.astype(np.float64) @ b.astype(np.float64)
    bound = 2 * k * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64))
    with backend() as be:
        assert np.all(np.abs(be.matmul(tensor(a), tensor(b)).numpy() - exact) <= bound)
        a[m - 1, k - 1] = np.nan
        got = be.matmul(tensor(a), tensor(b)).numpy()
    assert np.all(np.isnan(got[m - 1])) and np.all(np.abs(got[:m - 1] - exact[:m - 1]) <= bound[:m - 1])


@pytest.mark.parametrize("m,n,k", [(551, 2878, 52), (743, 2462, 127), (1153, 3201, 321),                     # 64 x 64
                                   (2003, 515, 66), (500, 2752, 97), (449, 2785, 193), (846, 1233, 200),     # 64 x 96
                                   (1096, 1943, 39), (961, 2690, 131), (705, 2753, 97), (1000, 2752, 256),   # 96 x 128
                                   (1000, 3083, 52), (1024, 3329, 129), (897, 3457, 159),                    # 128 x 128
                                   (513, 1345, 447), (481, 1441, 448), (1505, 385, 577), (129, 3361, 513)])  # 32 x 96
def test_matmul_on_bf16_pieces(m, n, k):
    """The tiles that multiply exact bf16 pieces: an element past a tile in rows and columns, K at and past their steps (32 and
    64), under the same bound.  Then operands that have no pieces, or whose small ones are lost: infinities and NaN give what
    the sum of the products gives, a tiny row and column (1e-36, against 1e30 and more) keep the bound."""
    rng = np.random.default_rng(m + n * k)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    a[3] *= np.float32(1e-36)
    b[:, n - 1] *= np.float32(1e-36)
    b[:, 5] *= np.float32(1e33)
    a[m - 1] *= np.float32(1e30)
    a[7] = 0.0
    exact = a.astype(np.float64) @ b.astype(np.float64)
    bound = 2 * k * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)) + k * 2.0 ** -149
    exact[m - 1, 5] = 0.0                                                   # beyond fp32
    with backend() as be:
        got = be.matmul(tensor(a), tensor(b)).numpy().astype(np.float64)
        got[m - 1, 5] = 0.0
        assert np.all(np.abs(got - exact) <= bound)
        a[0, 1], a[1, k - 1], b[0, 0] = np.inf, np.nan, -np.inf
        got = be.matmul(tensor(a), tensor(b)).numpy()
    assert np.all(np.isinf(got[0, 1:5])) and np.array_equal(np.sign(got[0, 1:5]), np.sign(b[1, 1:5])) and np.all(np.isnan(got[1]))
    assert np.array_equal(got[8:m - 1, 0], np.where(a[8:m - 1, 0] > 0, -np.inf, np.inf)) and np.isnan(got[7, 0])
    ok = (slice(8, m - 1), slice(6, n))
    assert np.all(np.abs(got[ok] - exact[ok]) <= bound[ok])


@pytest.mark.parametrize("m,n,k", [(551, 2878, 52), (500, 2752, 97), (1000, 2752, 256), (1000, 3083, 52), (1024, 3329, 129), (513, 1345, 447)])
def test_matmul_on_bf16_pieces_of_mixed_magnitudes(m, n, k):
    """Values whose small pieces are lost (2^-104 and below, fp32 subnormals) beside ordinary ones in a row or a column, where the
    other operand is zero at the ordinary ones and large at the small: the same bound; and no other output changes a bit."""
    rng = np.random.default_rng(m + n * k)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    with backend() as be:
        plain = be.matmul(tensor(a), tensor(b)).numpy().copy()
    rows, cols, ordinary = [2, 40, m - 1], [4, 70, n - 1], np.arange(k) % 5 == 0
    small = np.exp2(-104.0 - np.arange(k) % 24)
    for r, c, size in zip(rows, cols, (1.0, 1e-2, 2.0 ** -16)):            # (2^-144: subnormal)
        a[r], b[:, c] = np.where(ordinary, a[r], a[r] * small * size), np.where(ordinary, 0.0, b[:, c] * np.float32(1e30))
    a[9], b[:, 11] = np.where(ordinary, 0.0, a[9] * np.float32(1e30)), np.where(ordinary, b[:, 11], b[:, 11] * small)
    a[12], b[:, 17] = np.eye(1, k, 3), np.where(np.arange(k) == 3, 0.0, b[:, 17] * small)       # one ordinary product, by zero
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    bound = 2 * k * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64)) + k * 2.0 ** -149
    with backend() as be:
        got = be.matmul(tensor(a), tensor(b)).numpy()
    exact = a64 @ b64
    wrong = np.argwhere((np.abs(got - exact) > bound) & (np.abs(exact) < 1e38))                  # (row 9 by a column of 1e30: beyond fp32)
    assert not len(wrong), (wrong[:8], len(wrong))
    assert got[12, 17] == 0.0
    others = np.ones((m, n), bool)
    others[[*rows, 9, 12]], others[:, [*cols, 11, 17]] = False, False
    assert np.array_equal(got[others], plain[others])


@pytest.mark.parametrize("m,n,k", [(128, 1, 8500000), (1, (1 << 26) + 5, 3)])
def test_matmul_with_rows_beyond_32_bit_offsets(m, n, k):
    """A tile's rows of A, or a stage's rows of B, more than 4 GiB apart: what the last row and column hold is found there."""
    dev = DeviceBuffers()
    try:
        a, b, out = dev.alloc(m * k), dev.alloc(k * n), dev.alloc(m * n)
        three, five = dev.upload(np.array([3.0], np.float32)), dev.upload(np.array([5.0], np.float32))
        s = Stream().fill(a, 0, m * k).fill(b, 0, k * n)
        s.copy(three, a, 1, 0, m * k - 1).copy(five, b, 1, 0, k * n - 1).matmul(a, b, out, m, n, k).run()
        got = dev.download(out, (m * n,))
    finally:
        dev.release_all()
        HipNative.trim()
    assert got[-1] == 15.0 and np.count_nonzero(got) == 1


def test_matmul_rejects_shape_mismatch():                             # :80-86
    with backend() as be:
        with pytest.raises(ValueError, match="Shape mismatch"):
            be.matmul(tensor(rnd(3, 4, 3)), tensor(rnd(5, 2, 4)))


def test_elementwise_binary_ops():
    a, b = rnd(37, 53, 5), rnd(37, 53, 6) + 0.5
    with backend() as be:
        ta, tb = tensor(a), tensor(b)
        assert_close(ref.add(a, b), be.add(ta, tb), 1e-6, 1e-6)
        assert_close(ref.subtract(a, b), be.subtract(ta, tb), 1e-6, 1e-6)
        assert_close(ref.multiply(a, b), be.multiply(ta, tb), 1e-6, 1e-6)
        assert_close(ref.divide(a, b), be.divide(ta, tb), 1e-6, 1e-6)


def test_broadcast_and_scalar_ops_match_cpu():                        # :88-113
    a, row, col = rnd(8, 16, 100), rnd(1, 16, 101), rnd(8, 1, 102)
    with backend() as be:
        ta, tr, tc = tensor(a), tensor(row), tensor(col)
        assert_close(ref.add_row_vector(a, row), be.addRowVector(ta, tr))
        assert_close(ref.add_broadcast_cols(a, col), be.addBroadcastCols(ta, tc))
        assert_close(ref.subtract_broadcast_cols(a, col), be.subtractBroadcastCols(ta, tc))
        assert_close(ref.divide_broadcast_cols(a, col), be.divideBroadcastCols(ta, tc))
        assert_close(ref.multiply_broadcast_cols(a, col), be.multiplyBroadcastCols(ta, tc))
        assert_close(ref.multiply_broadcast_rows(a, row), be.multiplyBroadcastRows(ta, tr))
        assert_close(ref.add_scalar(a, 0.25), be.addScalar(ta, 0.25))
        assert_close(ref.divide_scalar(a, 1.5), be.divideScalar(ta, 1.5))
        assert_close(ref.multiply_scalar(a, -2.5), be.multiplyScalar(ta, -2.5))


@pytest.mark.parametrize("rows,cols", [(32, 24), (29, 513), (5, 2048), (1, 1)])
def test_reductions_and_transpose_match_cpu(rows, cols):              # :115-135 (+ wide rows :222-233)
    a = rnd(rows, cols, 111)
    with backend() as be:
        ta = tensor(a)
        assert_close(ref.transpose(a), be.transpose(ta))
        assert_close(ref.sum_rows(a), be.sumRows(ta))
        assert_close(ref.sum_along_rows(a), be.sumAlongRows(ta))
        assert_close(ref.sum_along_cols(a), be.sumAlongCols(ta))
        assert_close(ref.mean_along_rows(a), be.meanAlongRows(ta))
        assert_close(ref.variance_along_rows(a), be.varianceAlongRows(ta))
        assert_close(ref.max_along_rows(a), be.maxAlongRows(ta), 0, 0)
        # whole-tensor fp32 sums: the CPU's sequential sum itself carries ~n*eps relative error
        assert abs(ref.sum_(a) - be.sum(ta)) <= 1e-4 + 1e-5 * ref.sum_abs(a)
        assert abs(ref.sum_abs(a) - be.sumAbs(ta)) <= 1e-4 + 1e-5 * ref.sum_abs(a)


def test_unary_math_and_activations():
    a = rnd(19, 33, 7) * 10.0
    pos = np.abs(a) + 0.01
    with backend() as be:
        ta, tp = tensor(a), tensor(pos)
        assert_close(ref.sqrt(pos), be.sqrt(tp), 0, 1e-7)
        assert_close(ref.neg(a), be.neg(ta), 0, 0)
        assert_close(ref.exp(a), be.exp(ta), 0, 2e-7)
        assert_close(ref.log(pos), be.log(tp), 1e-7, 2e-7)
        assert_close(ref.tanh(a), be.tanh(ta), 1e-7, 2e-7)
        assert_close(ref.sigmoid(a), be.sigmoid(ta), 1e-7, 2e-7)
        assert_close(ref.relu(a), be.relu(ta), 0, 0)
        assert_close(ref.gelu(a), be.gelu(ta), 1e-6, 1e-6)
        g = rnd(19, 33, 8)
        assert_close(ref.relu_backward(a, g), be.reluBackward(ta, tensor(g)), 0, 0)
        assert_close(ref.gelu_backward(a, g), be.geluBackward(ta, tensor(g)), 1e-6, 1e-6)


def test_softmax_rows_matches_cpu_and_sums_to_one():
    for rows, cols, seed in [(32, 64, 11), (17, 769, 13), (3, 5000, 14)]:
        x = rnd(rows, cols, seed) * 20.0
        with backend() as be:
            p = be.softmaxRows(tensor(x)).numpy()
        assert_close(ref.softmax_rows(x), p, 1e-7, 1e-5)
        assert np.allclose(p.sum(1), 1.0, atol=1e-5)


def test_max_clamp_pow_and_scatter_add_rows_match_cpu():              # :137-172
    a = rnd(16, 20, 121)
    with backend() as be:
        ta = tensor(a)
        assert_close(ref.max_along_rows(a), be.maxAlongRows(ta))
        assert_close(ref.clamp(a, -0.25, 0.35), be.clamp(ta, -0.25, 0.35), 0, 0)
        assert_close(ref.pow_(a, 2.0), be.pow(ta, 2.0))
        for idx, ts, gs, tol in [([3, 1, 7, 2, 4, 5], 122, 123, 1e-4), ([3, 1, 7, 1, 4, 3], 124, 125, 1e-3)]:
            target_cpu = rnd(10, 8, ts)
            target_gpu = tensor(target_cpu)
            grad = rnd(6, 8, gs)
            ref.scatter_add_rows(target_cpu, idx, grad)
            Tensor.scatterAddRows(target_gpu, idx, tensor(grad))
            assert_close(target_cpu, target_gpu, tol, tol)


def test_scatter_add_rows_many_duplicates():                          # :174-197
    target_cpu = rnd(64, 32, 129)
    grad = rnd(128, 32, 130)
    idx = ref.JavaRandom(131).ints(128, 64)
    with backend():
        target_gpu = tensor(target_cpu)
        ref.scatter_add_rows(target_cpu, idx, grad)
        Tensor.scatterAddRows(target_gpu, list(idx), tensor(grad))
        assert_close(target_cpu, target_gpu, 1e-3, 1e-3)


def test_scalar_sum_abs_and_cross_entropy_loss_match_cpu():           # :199-238
    with backend() as be:
        a = rnd(23, 17, 126)
        assert abs(ref.sum_abs(a) - be.sumAbs(tensor(a))) <= 1e-4
        for rows, cols, ls, ts, tol in [(19, 31, 127, 128, 1e-4), (23, 777, 133, 134, 1e-3)]:
            logits = rnd(rows, cols, ls)
            targets = list(ref.JavaRandom(ts).ints(rows, cols))
            assert abs(ref.cross_entropy_loss(logits, targets) - be.crossEntropyLoss(tensor(logits), targets)) <= tol
        wide = rnd(29, 513, 132)
        assert abs(ref.sum_abs(wide) - be.sumAbs(tensor(wide))) <= 1e-3 + 1e-5 * ref.sum_abs(wide)


def test_softmax_backward_matches_cpu():                              # :240-266
    with backend() as be:
        for rows, cols, s1, s2 in [(32, 64, 10, 11), (17, 769, 12, 13)]:
            g, sm = rnd(rows, cols, s1), ref.softmax_rows(rnd(rows, cols, s2))
            assert_close(ref.softmax_backward(g, sm), be.softmaxBackward(tensor(g), tensor(sm)))
        with pytest.raises(ValueError, match="Shape mismatch"):       # :268-276
            be.softmaxBackward(tensor(rnd(2, 3, 21)), tensor(rnd(3, 2, 22)))


def test_layer_norm_backward_matches_cpu():                           # :278-323
    with backend() as be:
        for rows, cols, s1, s2 in [(16, 32, 31, 32), (11, 777, 33, 34)]:
            d, xh = rnd(rows, cols, s1), rnd(rows, cols, s2)
            std = (0.5 + np.abs(xh[:, :1])).astype(np.float32)
            assert_close(ref.layer_norm_backward(d, xh, std, cols),
                         be.layerNormBackward(tensor(d), tensor(xh), tensor(std), cols))
        with pytest.raises(ValueError, match="layerNormBackward: std"):
            be.layerNormBackward(tensor(rnd(4, 8, 41)), tensor(rnd(4, 8, 42)), tensor(rnd(4, 2, 43)), 8)


def test_cross_entropy_gradient_matches_cpu():                        # :325-372, at 1e-4 instead of 1e-3/1e-2
    with backend() as be:
        for rows, cols, ls, ts in [(32, 64, 51, 52), (17, 769, 53, 54)]:
            logits = rnd(rows, cols, ls)
            targets = list(ref.JavaRandom(ts).ints(rows, cols))
            assert_close(ref.cross_entropy_gradient(logits, targets),
                         be.crossEntropyGradient(tensor(logits), targets), 1e-6, 1e-4)
        with pytest.raises(ValueError, match="targets length"):
            be.crossEntropyGradient(tensor(rnd(4, 8, 61)), [0, 1, 2])


def test_cross_entropy_bad_target_gives_nan_not_a_fault():            # deepj_metal_jni.mm:472-476,497-503
    with backend() as be:
        g = be.crossEntropyGradient(tensor(rnd(2, 5, 1)), [1, 7]).numpy()
        assert np.all(np.isfinite(g[0])) and np.all(np.isnan(g[1]))


def test_adamw_update_matches_cpu_single_and_multiple_steps():        # :374-450
    lr, b1, b2, eps, wd = 1e-3, 0.9, 0.999, 1e-8, 0.01
    with backend() as be:
        w_cpu, g = rnd(32, 64, 71), rnd(32, 64, 72)
        mt_cpu, vt_cpu = np.zeros_like(w_cpu), np.zeros_like(w_cpu)
        w_gpu, mt_gpu, vt_gpu = tensor(w_cpu), Tensor(32, 64), Tensor(32, 64)
        ref.adamw_update(w_cpu, g, mt_cpu, vt_cpu, lr, b1, b2, eps, wd, 1 - b1, 1 - b2)
        be.adamWUpdate(w_gpu, tensor(g), mt_gpu, vt_gpu, lr, b1, b2, eps, wd, 1 - b1, 1 - b2)
        assert_close(w_cpu, w_gpu); assert_close(mt_cpu, mt_gpu); assert_close(vt_cpu, vt_gpu)

        w_cpu = rnd(16, 48, 81)
        mt_cpu, vt_cpu = np.zeros_like(w_cpu), np.zeros_like(w_cpu)
        w_gpu, mt_gpu, vt_gpu = tensor(w_cpu), Tensor(16, 48), Tensor(16, 48)
        for step in range(1, 6):
            g = rnd(16, 48, 90 + step)
            bc1 = np.float32(1.0) - np.float32(np.power(np.float64(np.float32(b1)), step))
            bc2 = np.float32(1.0) - np.float32(np.power(np.float64(np.float32(b2)), step))
            ref.adamw_update(w_cpu, g, mt_cpu, vt_cpu, lr, b1, b2, eps, wd, float(bc1), float(bc2))
            be.adamWUpdate(w_gpu, tensor(g), mt_gpu, vt_gpu, lr, b1, b2, eps, wd, float(bc1), float(bc2))
        assert_close(w_cpu, w_gpu); assert_close(mt_cpu, mt_gpu); assert_close(vt_cpu, vt_gpu)


def test_in_place_ops_and_chained_lazy_graph():
    a, b = rnd(9, 11, 200), rnd(9, 11, 201)
    with backend():
        t = tensor(a)
        t.addInPlace(tensor(b)).multiplyScalarInPlace(0.5).sigmoidInPlace().negInPlace()
        exp = ref.neg(ref.sigmoid(ref.multiply_scalar(ref.add(a, b), 0.5)))
        assert_close(exp, t, 1e-7, 1e-6)
        t.set(0, 0, 3.0)                       # host write -> re-upload on next use (Tensor.java:213-217)
        exp[0, 0] = 3.0
        assert_close(ref.add_scalar(exp, 1.0), t.addScalar(1.0), 1e-7, 1e-6)


def test_rmsnorm_composition_of_six_primitives():                     # RMSNorm1D.java:46-57 through primitive ops
    x, gamma = rnd(7, 256, 300), 1.0 + rnd(1, 256, 301)
    with backend():
        tx = tensor(x)
        rms = tx.multiply(tx).meanAlongRows().addScalar(1e-6).sqrt()
        out = tx.divideBroadcastCols(rms).multiplyBroadcastRows(tensor(gamma))
        assert_close(ref.rmsnorm(x, gamma), out, 1e-6, 1e-5)


# ── the boundary's failure behaviour, forced from the host ───────────────────

def test_native_errors_surface_as_exceptions_and_runtime_survives():
    HipNative.init(0)
    with pytest.raises(RuntimeError, match="Unknown op code in graph: 63"):    # deepj_metal_jni.mm:2120-2121
        HipNative.nativeFlushOps(np.array([63, 0, 0, 0], np.int32), 4)
    with pytest.raises(RuntimeError, match="Buffer not found for upload"):     # :1512-1516
        HipNative.nativeUploadBuffer(123456, np.zeros(4, np.float32))
    with pytest.raises(RuntimeError, match="Buffer not found for download"):   # :1528-1532
        HipNative.nativeDownloadBuffer(123456, np.zeros(4, np.float32))
    with pytest.raises(RuntimeError, match="missing GPU buffer id=999"):       # :1404-1410
        HipNative.nativeFlushOps(np.array([1, 999, 998, 997, 4], np.int32), 5)
    HipNative.nativeAllocBuffers([900001, 900002], [4, 2], 2)
    try:
        with pytest.raises(RuntimeError, match="holds 2 floats, op needs 4"):  # host-side bounds check
            HipNative.nativeFlushOps(np.array([8, 900001, 900002, 4], np.int32), 4)
        with pytest.raises(RuntimeError, match="truncated"):
            HipNative.nativeFlushOps(np.array([5, 900001, 900001], np.int32), 3)
        HipNative.nativeAllocBuffers([900001], [1 << 20], 1)                    # existing id: no-op (:1489)
        HipNative.nativeUploadBuffer(900001, np.arange(4, dtype=np.float32))
        out = np.zeros(4, np.float32)
        HipNative.nativeDownloadBuffer(900001, out)
        assert list(out) == [0, 1, 2, 3]
    finally:
        HipNative.nativeReleaseBuffers([900001, 900002, 424242], 3)             # unknown id ignored (:1545-1547)
    with backend() as be:                                                       # still works afterwards
        assert_close([[3.0]], be.add(tensor([[1.0]]), tensor([[2.0]])), 0, 0)


def test_graph_replay_is_refused_once_a_captured_buffer_or_the_workspace_is_gone():
    """A captured graph replays raw device addresses: after a buffer it names is released (or re-created elsewhere),
    or after the workspace it used was replaced by a larger one, a launch must fail and run nothing."""
    from deepj_amd.fused import DeviceBuffers, Stream
    HipNative.init(0)
    dev = DeviceBuffers()
    try:
        a, out = dev.upload(np.arange(8, dtype=np.float32)), dev.alloc(8)
        add = Stream().emit(op.OP_ADD_SCALAR, a, out, np.float32(1.0).view(np.int32), 8).array()
        g1 = HipNative.graphCapture(add)
        HipNative.graphLaunch(g1, 2)
        assert list(dev.download(out, (8,))) == [1, 2, 3, 4, 5, 6, 7, 8]
        dev.write(out, np.zeros(8, np.float32))
        dev.release(a)
        with pytest.raises(RuntimeError, match="released or reallocated"):
            HipNative.graphLaunch(g1, 1)
        assert not dev.download(out, (8,)).any(), "a refused replay must launch nothing"
        HipNative.graphDestroy(g1)
        # a graph that uses the workspace (normalised rows of an M > 1 Q8_LINEAR), then a stream that needs a larger one
        m, k, n = 8, 64, 4
        x, gm, w, o = dev.alloc(m * k), dev.alloc(k), dev.alloc(HipNative.q8Floats(k, n)), dev.alloc(m * n)
        Stream().fill(x, 0, m * k).fill(gm, 0, k).fill(w, 0, HipNative.q8Floats(k, n)).run()
        g2 = HipNative.graphCapture(Stream().q8_linear(x, w, o, m, k, n, gamma=gm).array())
        HipNative.graphLaunch(g2, 1)
        big_m, big_k = 16384, 8192                   # 128 Mi floats of normalised rows: more than any other test's stream needs
        bx, bg, bw, bo = (dev.alloc(big_m * big_k), dev.alloc(big_k), dev.alloc(HipNative.q8Floats(big_k, n)),
                          dev.alloc(big_m * n))
        Stream().fill(bx, 0, big_m * big_k).fill(bg, 0, big_k).fill(bw, 0, HipNative.q8Floats(big_k, n)).run()
        Stream().q8_linear(bx, bw, bo, big_m, big_k, n, gamma=bg).run()
        with pytest.raises(RuntimeError, match="workspace was reallocated"):
            HipNative.graphLaunch(g2, 1)
        HipNative.graphDestroy(g2)
        # opcode 82 once named an op that was withdrawn: it is an unknown opcode like any other
        with pytest.raises(RuntimeError, match="Unknown op code in graph: 82"):
            HipNative.nativeFlushOps(np.array([82, 2], np.int32), 2)
    finally:
        dev.release_all()


def test_released_buffers_are_recycled_without_new_driver_allocations():
    with backend() as be:
        t = tensor(rnd(64, 64, 1))
        for _ in range(3):
            t.addScalarInPlace(1.0)
            t.materialize()
        before = HipNative.poolStats()["driver_allocs"]
        for _ in range(50):
            t.addScalarInPlace(1.0)
            t.materialize()
        after = HipNative.poolStats()
        assert after["driver_allocs"] == before, "in-place rebinding must reuse pooled blocks"


@pytest.mark.parametrize("rows,cols", [(1, 1), (1, 5), (33, 4), (127, 32), (129, 36), (300, 1003), (1025, 192), (5, 2752)])
def test_column_sums_and_broadcasts_at_ragged_sizes(rows, cols):
    """sumRows with rows and columns that do not fill its 32 x 128 (or 32 x 32) passes: bound rows * 2^-24 * sum |a|.  The
    broadcasts give every value its own row's or column's operand: bit for bit."""
    rng = np.random.default_rng(rows * cols)
    a = rng.standard_normal((rows, cols)).astype(np.float32)
    row, col = rng.standard_normal((1, cols)).astype(np.float32), rng.standard_normal((rows, 1)).astype(np.float32)
    with backend() as be:
        t = tensor(a)
        got = be.sumRows(t).numpy()
        assert np.all(np.abs(got - a.sum(0, dtype=np.float64)) <= 2 * rows * 2.0 ** -24 * np.abs(a).sum(0, dtype=np.float64))
        assert np.array_equal(be.addRowVector(t, tensor(row)).numpy(), a + row)
        assert np.array_equal(be.multiplyBroadcastRows(t, tensor(row)).numpy(), a * row)
        assert np.array_equal(be.subtractBroadcastCols(t, tensor(col)).numpy(), a - col)
        assert np.array_equal(be.divideBroadcastCols(t, tensor(col)).numpy(), a / col)


def test_adamw_steps_recorded_together_match_steps_one_by_one():
    """More tensors than one launch takes, odd sizes, and a parameter stepped twice in the same flush (which must see its
    first step)."""
    rng = np.random.default_rng(3)
    shapes = [(1, n) for n in (1, 2, 3, 5, 7, 64, 255, 1001)] + [(33, 17)] * 11
    hyper = (1e-2, 0.9, 0.999, 1e-8, 0.01, 0.1, 0.001)
    results = []
    for flush_each in (False, True):
        rng = np.random.default_rng(3)
        with backend() as be:
            sets = [[tensor(np.abs(rng.standard_normal(s)).astype(np.float32)) for _ in range(4)] for s in shapes]
            for k in list(range(len(sets))) + [2]:
                be.adamWUpdate(*sets[k], *hyper)
                if flush_each:
                    be.graph.flush()
            results.append([t.numpy().copy() for four in sets for t in four])
    assert all(np.array_equal(x, y) for x, y in zip(*results))
