"""The Q8 GEMM that multiplies a batch of rows straight from the int8 weights, through the C ABI against float64 on the
oracle's dequantised weights, at the edges of its tiles (32 or 64 rows and columns), of its 128-k chunks and of the ways it
deals them: one to four wavefronts with work, K shared by several workgroups, odd and ragged everything.

Gate on the rms error of the whole product: activations and weights are held exactly, and an output is at most four sums (one a
wavefront) of G = K / 128 scaled group sums, whose n-th rounding is 2^-24 of a partial sum of n groups: 2^-23 (1 + sqrt(G / 2))
of the product's rms covers that and the roundings inside a group."""
import numpy as np
import pytest

from deepj_amd import HipNative, JavaRandom
from deepj_amd.fused import DeviceBuffers, Stream
from oracle import cpu_ref as ref

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    d = DeviceBuffers()
    yield d
    d.release_all()


def check(got, exp, k, what, times=1):
    size = np.sqrt(np.mean(exp ** 2, axis=1, keepdims=True))
    assert not got[size[:, 0] == 0].any(), f"{what}: a row of zeros"
    err = float(np.sqrt(np.mean(((got - exp) / np.where(size == 0, 1, size)) ** 2)))
    assert err <= times * 2.0 ** -23 * (1 + np.sqrt(k / 256)), f"{what}: rms error {err:.2e}"


def rms_normalised(x, gamma):
    return x / np.sqrt((x * x).mean(1, keepdims=True) + 1e-6) * gamma


# Products that k_gemm_q8 keeps, under the same gate (its sums are no longer): eight, seven and eight workgroups sharing K, and
# small weights without a normalisation in front
ON_K_GEMM_Q8 = [(30, 11008, 1024, 0), (5, 5600, 2050, 0), (200, 12300, 500, 0), (40, 96, 50001, 0), (250, 288, 20002, 0)]


@pytest.mark.parametrize("m,k,n,norm", [(2, 32, 2, 1), (7, 31, 33, 1), (32, 128, 32, 1), (33, 129, 31, 1), (64, 160, 65, 1), (65, 416, 64, 1), (96, 512, 97, 1),
                                        (31, 640, 127, 1), (30, 11008, 1023, 0), (200, 1028, 5002, 0), (30, 1100, 24497, 0), (50, 1100, 24497, 0), *ON_K_GEMM_Q8])
def test_product_at_the_edges(dev, m, k, n, norm):
    assert (HipNative.q8GemmRowsTile(m, k, n, norm)[0] == 0) == ((m, k, n, norm) in ON_K_GEMM_Q8)
    w, x, gamma = JavaRandom(5).tensor(k, n, k ** -0.5), JavaRandom(6).tensor(m, k, 1.0), JavaRandom(7).tensor(1, k, 1.0)
    if m > 4:
        x[1] = 0.0                                       # a row without a largest value
        x[2] *= 1e-18                                    # rows far from one, which leave the others as they are
        x[3] *= 1e15
    src, wq, xb, ob, gb = dev.upload(w), dev.alloc(HipNative.q8Floats(k, n)), dev.upload(x), dev.alloc(m * n), dev.upload(gamma)
    Stream().q8_quantize(src, wq, k, n).run()
    op = Stream().q8_linear(xb, wq, ob, m, k, n, gamma=gb if norm else -1)
    op.run()
    got = dev.download(ob, (m, n)).copy()
    op.run()
    assert np.array_equal(got, dev.download(ob, (m, n)))                 # the same bits again
    dev.release(src, wq, xb, ob, gb)
    a = rms_normalised(x.astype(np.float64), gamma) if norm else x.astype(np.float64)
    check(got, a @ ref.q8_roundtrip(w).astype(np.float64), k, f"{m} x {k} x {n}", times=1 + norm)


# (tile rows, tile columns, workgroups that share its K), every one of them: K of whole chunks, whose scales come in one load, and
# ragged, whose scales come group by group; columns that end inside a tile
EVERY_TILE = [((32, 32, 1), (2, 128, 33, 1)), ((32, 32, 1), (2, 40, 33, 1)), ((32, 32, 2), (30, 3072, 2050, 1)), ((32, 32, 2), (30, 3000, 2050, 1)),
              ((32, 32, 4), (2, 1152, 250, 1)), ((32, 32, 4), (2, 1028, 250, 1)), ((32, 64, 1), (640, 640, 500, 1)), ((32, 64, 1), (640, 600, 500, 1)),
              ((32, 64, 2), (640, 2048, 1002, 1)), ((32, 64, 2), (640, 3000, 1002, 1)), ((32, 64, 4), (200, 4096, 1500, 1)), ((32, 64, 4), (700, 6004, 500, 1)),
              ((32, 96, 1), (400, 1152, 1500, 1)), ((32, 96, 1), (400, 1028, 1500, 1)), ((64, 32, 1), (33, 256, 6150, 1)), ((64, 32, 1), (33, 200, 6150, 1)),
              ((64, 64, 1), (700, 512, 3010, 1)), ((64, 64, 1), (700, 416, 3010, 1)), ((64, 64, 2), (130, 6144, 2050, 1)), ((64, 64, 2), (130, 6004, 2050, 1)),
              ((64, 96, 1), (640, 1152, 2049, 1)), ((64, 96, 1), (640, 1028, 2049, 1))]


@pytest.mark.parametrize("tile,shape", EVERY_TILE)
def test_product_on_every_tile(dev, tile, shape):
    assert HipNative.q8GemmRowsTile(*shape) == tile
    test_product_at_the_edges(dev, *shape)


@pytest.mark.parametrize("m,k,n,there", [(128, 6144, 4096, 1.26e-7), (250, 8224, 2050, 1.68e-7), (96, 2048, 6144, 1.12e-7)])
def test_error_is_no_larger_than_the_kernel_it_stands_in_for(dev, m, k, n, there):
    """`there`: k_gemm_q8's rms error on the same product, with the numbers of other seeds 1 % apart."""
    assert HipNative.q8GemmRowsTile(m, k, n)[0]
    w, x = JavaRandom(5).tensor(k, n, k ** -0.5), JavaRandom(6).tensor(m, k, 1.0)
    src, wq, xb, ob = dev.upload(w), dev.alloc(HipNative.q8Floats(k, n)), dev.upload(x), dev.alloc(m * n)
    Stream().q8_quantize(src, wq, k, n).q8_linear(xb, wq, ob, m, k, n).run()
    got = dev.download(ob, (m, n)).copy()
    dev.release(src, wq, xb, ob)
    exp = x.astype(np.float64) @ ref.q8_roundtrip(w).astype(np.float64)
    err = float(np.sqrt(np.mean((got - exp) ** 2) / np.mean(exp ** 2)))
    assert err <= 1.01 * there, f"rms error {err:.3e}"


@pytest.mark.parametrize("m,k,n,norm", [(30, 2048, 5632, 0), (96, 4096, 4500, 0), (64, 4096, 6000, 1), (30, 11008, 1023, 0), (7, 12320, 1500, 1)])
@pytest.mark.parametrize("spread", ["outlier", "groups"])
def test_the_range_within_a_row_costs_no_bits(dev, m, k, n, norm, spread):
    """A column of 1e4 to 1e8 whose weights are zero, and 32-k groups over twelve decades whose weights run the other way: an
    activation's bits are its own, whatever the largest of its row is."""
    assert HipNative.q8GemmRowsTile(m, k, n, norm)[0]
    rng = np.random.default_rng(k + norm)
    w, x, gamma = (rng.standard_normal(s).astype(np.float32) for s in ((k, n), (m, k), (1, k)))
    by = np.ones(k, np.float32)
    if spread == "outlier":
        w[33] = 0.0
        by[33] = 1e8
        x[: m // 2, 33] *= np.float32(1e-4)
    else:
        by[:] = np.repeat(10.0 ** rng.uniform(-6, 6, (k + 31) // 32), 32)[:k]
        w /= by[:, None]
    if norm:
        gamma *= by                                      # (the normalised row has the range)
    else:
        x *= by
    src, wq, xb, ob, gb = dev.upload(w), dev.alloc(HipNative.q8Floats(k, n)), dev.upload(x), dev.alloc(m * n), dev.upload(gamma)
    Stream().q8_quantize(src, wq, k, n).q8_linear(xb, wq, ob, m, k, n, gamma=gb if norm else -1).run()
    got = dev.download(ob, (m, n)).copy()
    dev.release(src, wq, xb, ob, gb)
    a = rms_normalised(x.astype(np.float64), gamma) if norm else x.astype(np.float64)
    check(got, a @ ref.q8_roundtrip(w).astype(np.float64), k, f"{m} x {k} x {n} {spread}", times=1 + norm)


# (on: the ones that run here; the others on k_gemm_q8.)  The last but two: K shared, the epilogue in the sum of the shares
EPILOGUES = ("bias_gelu_residual", "swiglu", "rms", "layernorm")


@pytest.mark.parametrize("m,k,n,on", [(9, 200, 46, EPILOGUES[2:]), (64, 2052, 2100, ()), (30, 8224, 1026, EPILOGUES[2:]), (250, 8224, 2050, EPILOGUES),
                                      (200, 1028, 5002, EPILOGUES), (40, 2056, 4100, EPILOGUES[1:2])])
@pytest.mark.parametrize("epilogue", EPILOGUES)
def test_prologues_and_epilogues(dev, m, k, n, on, epilogue):
    sw = epilogue == "swiglu"
    assert (HipNative.q8GemmRowsTile(m, k, n * (1 + sw), epilogue in EPILOGUES[2:])[0] > 0) == (epilogue in on)
    w, x = [JavaRandom(7 + i).tensor(k, n, k ** -0.5) for i in range(1 + sw)], JavaRandom(9).tensor(m, k, 1.0)
    vec = [JavaRandom(10 + i).tensor(1, k if i > 1 else n, 0.5) for i in range(4)]
    res = JavaRandom(15).tensor(m, n, 1.0)
    wq, xb, ob, rb = dev.alloc(HipNative.q8Floats(k, n * (1 + sw))), dev.upload(x), dev.alloc(m * n), dev.upload(res)
    vb = [dev.upload(v) for v in vec]
    for i, wi in enumerate(w):
        src = dev.upload(wi)
        Stream().q8_quantize(src, wq, k, n, i, 1 + sw, n * (1 + sw)).run()
        dev.release(src)
    kw = {"bias_gelu_residual": dict(bias=vb[0], gelu=True, residual=rb), "swiglu": dict(swiglu=True, bias=vb[0], bias2=vb[1]),
          "rms": dict(gamma=vb[2]), "layernorm": dict(gamma=vb[2], beta=vb[3], bias=vb[0])}[epilogue]
    Stream().q8_linear(xb, wq, ob, m, k, n, **kw).run()
    got = dev.download(ob, (m, n)).copy()
    dev.release(wq, xb, ob, rb, *vb)
    a, v, deq = x.astype(np.float64), [t.astype(np.float64) for t in vec], [ref.q8_roundtrip(wi).astype(np.float64) for wi in w]
    if epilogue == "rms":
        a = rms_normalised(a, v[2])
    if epilogue == "layernorm":
        c = a - a.mean(1, keepdims=True)
        a = c / np.sqrt((c * c).mean(1, keepdims=True) + 1e-5) * v[2] + v[3]
    y = a @ deq[0]
    if epilogue == "bias_gelu_residual":
        y = y + v[0]
        y = res + 0.5 * y * (1 + np.tanh(0.7978845608 * (y + 0.044715 * y ** 3)))
    if sw:
        gate, up = y + v[0], a @ deq[1] + v[1]
        y = gate / (1 + np.exp(-gate)) * up
    if epilogue == "layernorm":
        y = y + v[0]
    # (the normalisations and activations add some roundings of their own: as much again)
    check(got, y, k, epilogue, times=2)


@pytest.mark.parametrize("m,k,n,taken", [(40, 600, 8000, False), (40, 2048, 8000, True)])
def test_a_row_that_is_not_finite_stays_alone(dev, m, k, n, taken):
    assert (HipNative.q8GemmRowsTile(m, k, n)[0] > 0) == taken           # k_gemm_q8 the other one
    w, x = JavaRandom(5).tensor(k, n, 0.05), JavaRandom(6).tensor(m, k, 1.0)
    src, wq, xb, ob = dev.upload(w), dev.alloc(HipNative.q8Floats(k, n)), dev.upload(x), dev.alloc(m * n)
    op = Stream().q8_quantize(src, wq, k, n).q8_linear(xb, wq, ob, m, k, n)
    op.run()
    clean = dev.download(ob, (m, n)).copy()
    x[3, 17], x[35, 599] = np.inf, np.nan
    dev.write(xb, x)
    op.run()
    got = dev.download(ob, (m, n)).copy()
    dev.release(src, wq, xb, ob)
    assert not np.isfinite(got[[3, 35]]).any()
    keep = [r for r in range(m) if r not in (3, 35)]
    assert np.array_equal(got[keep], clean[keep])


@pytest.mark.parametrize("widths,last_alone", [((64, 512, 50000, 64), False), ((1500, 512, 512, 64), True), ((2048, 1000, 2048, 64), False)])
def test_products_in_a_row_have_the_same_bits_whatever_the_block_of_pieces_holds(dev, widths, last_alone):
    """Three products behind one another, each multiplying the rows of the one in front as they are: the third takes the kernel that
    it takes with its pieces made (also where it takes another by itself), in the first run, which makes the block, as after a
    larger one; with its pieces behind the second one's and, where those lie far enough in, in front of them."""
    m, makes_block = 100, widths[2] == 50000
    rng = np.random.default_rng(3)
    assert [HipNative.q8GemmRowsTile(m, k, n, norm=k == widths[0])[0] > 0 for k, n in zip(widths, widths[1:])] == [True, True, last_alone]
    weights, rows = [], [dev.upload(rng.standard_normal((m, widths[0])).astype(np.float32)), *(dev.alloc(m * n) for n in widths[1:])]
    gamma, big_m, big_k, big_n = dev.upload(np.ones(widths[0], np.float32)), 512, 16384, 1026
    for k, n in (*zip(widths, widths[1:]), (big_k, big_n)):
        last = rng.standard_normal((k, n), dtype=np.float32) * np.float32(k ** -0.5)
        if len(weights) == 2:
            third = last
        src = dev.upload(last)
        weights.append(dev.alloc(HipNative.q8Floats(k, n)))
        Stream().q8_quantize(src, weights[-1], k, n).run()
        dev.release(src)
    big_x, big_o = dev.alloc(big_m * big_k), dev.alloc(big_m * big_n)
    three, big = Stream(), Stream().fill(big_x, 0, big_m * big_k).q8_linear(big_x, weights[3], big_o, big_m, big_k, big_n)
    for i, (k, n) in enumerate(zip(widths, widths[1:])):
        three.q8_linear(rows[i], weights[i], rows[i + 1], m, k, n, gamma=-1 if i else gamma)
    driver_allocs = lambda: HipNative.poolStats()["driver_allocs"]
    before = driver_allocs()
    three.run()
    made = driver_allocs()
    first = dev.download(rows[3], (m, widths[3])).copy()
    check(first, dev.download(rows[2], (m, widths[2])).astype(np.float64) @ ref.q8_roundtrip(third).astype(np.float64), widths[2], widths)
    big.run()
    if makes_block:
        assert before < made < driver_allocs()                           # a block of the size that the three need, then a larger one
    Stream().fill(rows[3], 0, m * widths[3]).run()
    three.run()
    assert np.array_equal(dev.download(rows[3], (m, widths[3])), first)
    dev.release(*weights, *rows, gamma, big_x, big_o)


def test_a_captured_product_outlives_a_larger_one(dev):
    """A product without a normalisation needs no workspace: a graph of it stays launchable whatever other streams need, over the
    block of pieces that it was captured with, also beside graphs of other blocks and once one of its own block is gone."""
    m, k, n = 30, 2048, 6144
    big_m, big_k, big_n = 767, 32768, 2050               # 41 Mi floats of pieces and partial products: more than any other test's
    assert HipNative.q8GemmRowsTile(m, k, n)[0] and HipNative.q8GemmRowsTile(big_m, big_k, big_n)[0]
    w, x = JavaRandom(5).tensor(k, n, k ** -0.5), JavaRandom(6).tensor(m, k, 1.0)
    src, wq, xb, ob = dev.upload(w), dev.alloc(HipNative.q8Floats(k, n)), dev.upload(x), dev.alloc(m * n)
    Stream().q8_quantize(src, wq, k, n).run()
    words = Stream().q8_linear(xb, wq, ob, m, k, n)
    words.run()
    expected = dev.download(ob, (m, n)).copy()
    big_x, big_w, big_o = dev.alloc(big_m * big_k), dev.alloc(HipNative.q8Floats(big_k, big_n)), dev.alloc(big_m * big_n)
    Stream().fill(big_x, 0, big_m * big_k).fill(big_w, 0, HipNative.q8Floats(big_k, big_n)).run()
    graphs = [HipNative.graphCapture(words.array()) for _ in range(2)]

    def replays(graph):
        for _ in range(3):
            dev.write(ob, np.zeros((m, n), np.float32))
            HipNative.graphLaunch(graph, 2)
            assert np.array_equal(dev.download(ob, (m, n)), expected)

    allocs = HipNative.poolStats()["driver_allocs"]
    Stream().q8_linear(big_x, big_w, big_o, big_m, big_k, big_n).run()
    assert HipNative.poolStats()["driver_allocs"] == allocs + 1
    graphs.append(HipNative.graphCapture(words.array()))
    for g in (0, 2, 1):
        replays(graphs[g])
        HipNative.graphDestroy(graphs[g])
    dev.release(src, wq, xb, ob, big_x, big_w, big_o)


@pytest.mark.parametrize("m,k,n,n2,norm", [(90, 768, 768, 3072, "layer"), (75, 1024, 1024, 2304, "rms"), (33, 2752, 1000, 2000, "rms"), (64, 1024, 772, 3000, "layer"),
                                           (2, 768, 516, 2048, "rms"), (200, 1100, 768, 2304, "layer"), (65, 4096, 1028, 3001, "rms")])
def test_a_product_that_shares_k_leaves_the_next_ones_pieces_without_changing_a_bit(dev, m, k, n, n2, norm):
    """The sum of k_gemm_q8's shares also normalises and splits the rows for the product behind it: the bits of the two ops by
    themselves, with a ragged batch, widths past a whole chunk, both norms; another gain in between and the second splits its own."""
    rng = np.random.default_rng(m + n)
    f = lambda *s: rng.standard_normal(s).astype(np.float32)
    assert HipNative.q8GemmRowsTile(m, n, n2, norm=True)[0] and not HipNative.q8GemmRowsTile(m, k, n)[0]

    def q8(r, c):
        src, dst = dev.upload(f(r, c) * np.float32(r ** -0.5)), dev.alloc(HipNative.q8Floats(r, c))
        Stream().q8_quantize(src, dst, r, c, 0, 1, c).run()
        return dst
    w1, w2 = q8(k, n), q8(n, n2)
    x, res, bias, gamma, beta = dev.upload(f(m, k)), dev.upload(f(m, n)), dev.upload(f(1, n)), dev.upload(1 + 0.1 * f(1, n)), dev.upload(0.1 * f(1, n))
    mid, out = dev.alloc(m * n), dev.alloc(m * n2)
    norms = dict(gamma=gamma, beta=beta) if norm == "layer" else dict(gamma=gamma)
    first = Stream().q8_linear(x, w1, mid, m, k, n, bias=bias, residual=res)
    second = Stream().q8_linear(mid, w2, out, m, n, n2, **norms)
    first.run(), second.run()
    want = dev.download(mid, (m, n)), dev.download(out, (m, n2))
    both = Stream()
    both.words = first.words + second.words
    for _ in range(2):
        Stream().fill(mid, 0, m * n).fill(out, 0, m * n2).run()
        both.run()
        assert np.array_equal(dev.download(mid, (m, n)), want[0]) and np.array_equal(dev.download(out, (m, n2)), want[1])
    alone = [int(HipNative.profileOps(s.array(), 2, detail=True)[2][0]) for s in (first, second)]
    together = [int(c) for c in HipNative.profileOps(both.array(), 2, detail=True)[2]]
    if alone[0] > 1:                                              # (it shares its K here)
        assert together == [alone[0], alone[1] - 1], (alone, together)
    handle = HipNative.graphCapture(both.array())
    for _ in range(3):
        Stream().fill(mid, 0, m * n).fill(out, 0, m * n2).run()
        HipNative.graphLaunch(handle)
        assert np.array_equal(dev.download(out, (m, n2)), want[1])
    HipNative.graphDestroy(handle)
    other = Stream().q8_linear(mid, w2, out, m, n, n2, **dict(norms, gamma=bias))
    both.words = first.words + Stream().fill(out, 0, m * n2).words + other.words
    both.run()
    apart = dev.download(out, (m, n2))
    other.run()
    assert np.array_equal(dev.download(out, (m, n2)), apart)


@pytest.mark.parametrize("m,d,dff,gated", [(64, 2048, 5632, True), (30, 2048, 5632, True), (90, 768, 3072, False), (75, 1024, 2752, True), (16, 256, 688, True),
                                           (33, 512, 1001, False), (2, 768, 2050, True), (65, 512, 1100, True), (40, 768, 1003, True), (200, 1024, 4104, False)])
def test_a_feed_forward_layer_hands_its_hidden_rows_on_in_pieces(dev, m, d, dff, gated):
    """The hidden rows' product leaves them for the one behind it in operand order: both outputs against float64, the first one's bits
    as by itself, in a captured graph too; ragged batches and widths (rows up to a multiple of 32 and columns up to a whole
    chunk are zeros there, whatever the memory held), and the layer's next product, which takes its pieces from a third place."""
    rng = np.random.default_rng(m + dff)
    f = lambda *s: rng.standard_normal(s).astype(np.float32)

    def q8(*parts):
        dst, r, c = dev.alloc(HipNative.q8Floats(parts[0].shape[0], parts[0].shape[1] * len(parts))), *parts[0].shape
        for i, p in enumerate(parts):
            src = dev.upload(p)
            Stream().q8_quantize(src, dst, r, c, i, len(parts), c * len(parts)).run()
            dev.release(src)
        return dst
    ups = [f(d, dff) * np.float32(d ** -0.5) for _ in range(2 if gated else 1)]
    wd, wq = f(dff, d) * np.float32(dff ** -0.5), f(d, 3 * d) * np.float32(d ** -0.5)
    x, gamma, bias = f(m, d), 1 + 0.1 * f(d), 0.1 * f(dff)
    w1, w2, w3 = q8(*ups), q8(wd), q8(wq)
    xb, gb, bb = dev.upload(x), dev.upload(gamma), dev.upload(bias)
    hidden, out, last = dev.alloc(m * dff), dev.alloc(m * d), dev.alloc(m * 3 * d)
    tiles = HipNative.q8GemmRowsTile(m, d, len(ups) * dff, norm=True)
    assert tiles[0]
    behind, by_itself = HipNative.q8GemmRowsTileBehind(m, dff, d), HipNative.q8GemmRowsTile(m, dff, d)
    first = Stream().q8_linear(xb, w1, hidden, m, d, dff, gamma=gb, bias=bb, bias2=bb if gated else -1, swiglu=gated, gelu=not gated)
    second = Stream().q8_linear(hidden, w2, out, m, dff, d, residual=xb)
    third = Stream().q8_linear(out, w3, last, m, d, 3 * d, gamma=gb)
    first.run()
    hidden_alone = dev.download(hidden, (m, dff))
    layer = Stream()
    layer.words = first.words + second.words + third.words
    poison, poison_out = dev.upload(np.full((700, dff), np.nan, np.float32)), dev.alloc(700 * d)

    def results():
        return dev.download(hidden, (m, dff)), dev.download(out, (m, d)), dev.download(last, (m, 3 * d))
    layer.run()                                                   # (sizes the scratch)
    Stream().q8_linear(poison, w2, poison_out, 700, dff, d).run()
    Stream().fill(hidden, 0, m * dff).fill(out, 0, m * d).fill(last, 0, m * 3 * d).run()
    Stream().fill(poison, 0, 700 * dff).fill(poison_out, 0, 700 * d).run()       # (a later buffer may get the memory)
    layer.run()
    got = results()
    assert np.array_equal(got[0], hidden_alone)
    # the second one runs on the kernel that it is said to take, its rows ready, and has that kernel's bits
    launches = [int(c) for c in HipNative.profileOps(layer.array(), 2, detail=True)[2]]
    if tiles[2] == 1 and behind[0]:
        assert launches[1] == (1 if behind[2] == 1 else 2), (launches, behind)
    if tiles[2] > 1 or not behind[0] or behind == by_itself:
        second.run()
        assert np.array_equal(dev.download(out, (m, d)), got[1])
    deq = lambda w: ref.q8_roundtrip(w).astype(np.float64)
    check(got[1], got[0].astype(np.float64) @ deq(wd) + x, dff, f"{m} x {d} over {dff}")
    check(got[2], rms_normalised(got[1].astype(np.float64), gamma) @ deq(wq), d, f"{m} x {3 * d} over {d}", times=2)      # (and the normalisation's roundings)
    graph = HipNative.graphCapture(layer.array())
    for _ in range(3):
        Stream().fill(hidden, 0, m * dff).fill(out, 0, m * d).fill(last, 0, m * 3 * d).run()
        HipNative.graphLaunch(graph)
        assert all(np.array_equal(a, b) for a, b in zip(results(), got))
    HipNative.graphDestroy(graph)
    dev.release(w1, w2, w3, xb, gb, bb, hidden, out, last, poison, poison_out)


@pytest.mark.parametrize("m,k,n,norm,gated", [(17, 1536, 12288, True, False), (32, 1500, 32768, True, True), (20, 4096, 9216, False, False), (31, 2048, 11264, False, True)])
def test_17_to_32_rows_read_the_int8_weights_whatever_copies_there_are(dev, m, k, n, norm, gated):
    """Its bits with a copy in place are those without one; a captured stream then outlives the copy."""
    rng = np.random.default_rng(m + n)
    f = lambda *s: rng.standard_normal(s).astype(np.float32)
    assert HipNative.q8GemmTilePrepared(m, k, n)[0]
    src, wq = dev.upload(f(k, n) * np.float32(k ** -0.5)), dev.alloc(HipNative.q8Floats(k, n))
    Stream().q8_quantize(src, wq, k, n, 0, 1, n).run()
    x, g, out, n_out = dev.upload(f(m, k)), dev.upload(1 + 0.1 * f(k)), dev.alloc(m * n), n // 2 if gated else n
    s = Stream().q8_linear(x, wq, out, m, k, n_out, gamma=g if norm else -1, swiglu=gated)
    s.run()
    want = dev.download(out, (m, n_out))
    copy = dev.alloc(HipNative.q8PreparedFloats(k, n))
    Stream().q8_prepare(wq, copy, k, n).fill(out, 0, m * n_out).run()
    s.run()
    assert np.isfinite(want).all() and np.array_equal(dev.download(out, (m, n_out)), want)
    graph = HipNative.graphCapture(s.array())
    dev.release(copy)
    for _ in range(3):
        Stream().fill(out, 0, m * n_out).run()
        HipNative.graphLaunch(graph)
        assert np.array_equal(dev.download(out, (m, n_out)), want)
    HipNative.graphDestroy(graph)
    dev.release(src, wq, x, g, out)
