"""Runs of tokens as one launch (deepj_hip_token_plan_*) against the launches of a token and the prompt's rows: every way the
work is dealt to groups and workgroups, at the edges of its tiles, slices, key splits and item slots."""
import ctypes as C
import time

import numpy as np
import pytest

from deepj_amd import models, GPTConfig, GPTModel, HipNative, LlamaConfig, LlamaModel, TextGenerator, parameter_names, parameter_shapes
from deepj_amd import opcodes as op
from deepj_amd._native import library
from deepj_amd.fused import Stream
from oracle import cpu_ref as ref

pytestmark = pytest.mark.gpu


def model(gpt, vocab, max_seq, d, heads, layers, dff, groups, seed=7, **changed):
    """Drawn weights; `changed`: a weight's name (with __ for its dot) and what makes its values from the drawn ones."""
    cfg = (GPTConfig if gpt else LlamaConfig)(vocab, max_seq, d, heads, layers, dff)
    m = (GPTModel if gpt else LlamaModel)(cfg, None)
    m.setTokenGroups(groups)
    rng = np.random.default_rng(seed)
    for name, (r, c) in zip(parameter_names(cfg), parameter_shapes(cfg)):
        a = rng.standard_normal((r, c), dtype=np.float32) * np.float32(d ** -0.5)
        a = 1.0 + a if name.split(".")[-1] in ("g1", "g2", "gf") else a
        m.setWeight(name, changed.get(name.replace(".", "__"), lambda v: v)(a))
    m.finalize()
    return m


def plan_of(m):
    return library().deepj_runner_token_plan(m._h)


# (gpt, vocab, d, heads, dff, groups, prompt): one to eight groups with even and uneven heads and hidden units; widths that leave
# workgroups without a tile (64, 96), a last tile of one word, hidden widths no multiple of 64, 8 or 4; all head widths; one key to
# several rounds of key tiles; wavefronts with more items than slots (2048 over 8192 on four groups, 4096); rows of two sets; heads of
# several passes, and of none in most workgroups; more weights than the memory-side cache holds (4096 over 11008 with 60000 words)
SHAPES = [(False, 251, 64, 2, 50, 1, 3), (False, 17001, 64, 2, 50, 1, 20), (True, 33000, 128, 2, 300, 2, 9), (False, 97, 96, 3, 130, 2, 60), (True, 253, 64, 2, 173, 2, 5), (False, 4097, 256, 8, 697, 1, 30),
          (False, 300, 256, 8, 697, 8, 30), (True, 1003, 320, 10, 1000, 4, 70), (True, 300, 384, 6, 1537, 4, 200), (False, 64, 128, 4, 260, 4, 1),
          (False, 500, 640, 5, 1000, 4, 900), (True, 1000, 768, 12, 3072, 8, 130), (False, 300, 512, 16, 1376, 1, 1500),
          (False, 8193, 1024, 16, 2752, 8, 1100), (False, 300, 2048, 16, 8192, 4, 40), (False, 2000, 2112, 33, 5000, 8, 40),
          (False, 500, 4096, 32, 11008, 8, 20), (False, 60000, 4096, 32, 11008, 8, 20)]


@pytest.mark.parametrize("gpt,vocab,d,heads,dff,groups,prompt", SHAPES)
def test_tokens_of_a_run_equal_those_of_launches(gpt, vocab, d, heads, dff, groups, prompt):
    """Stepped logits against the prompt's rows (the tolerance of the other such tests, of logits of order 1 to 5), a greedy run
    against the launches' and the prompt's largest logit, a sampled one, and one that takes turns with launches."""
    new = 12
    m = model(gpt, vocab, prompt + 40, d, heads, 2, dff, groups)
    try:
        assert plan_of(m) and library().deepj_hip_token_plan_groups(plan_of(m)) == groups
        ids = ref.JavaRandom(5).ints(prompt + new, vocab)
        full = m.forward(ids)
        scale = max(1.0, float(np.abs(full).max()) / 5)
        m.reset()
        m.prefill(ids[:prompt], choose_next=False)
        for t in range(prompt, prompt + new):
            m.step(int(ids[t]))
            assert float(np.max(np.abs(m.lastLogits() - full[t]))) <= 2e-4 * scale, t
        greedy = TextGenerator.generate(m, ids[:prompt], 30, top_k=1)
        logits = m.forward(greedy)
        for t in range(prompt, len(greedy)):
            assert logits[t - 1].max() - logits[t - 1, greedy[t]] <= 4e-4 * scale, t
        assert np.array_equal(greedy, TextGenerator.generate(m, ids[:prompt], 30, top_k=1))
        assert np.array_equal(greedy, TextGenerator.generate(m, ids[:prompt], 30, top_k=1, use_graph=False))
        sampled = [TextGenerator.generate(m, ids[:prompt], 20, 0.9, 5, 3, use_graph=g) for g in (True, False)]
        assert np.array_equal(*sampled)
        m.reset()
        m.prefill(ids[:prompt])
        for n, graph in ((5, True), (3, False), (1, True), (7, True), (2, False), (11, True)):
            m.decode(n, use_graph=graph)
        assert np.array_equal(m.tokens(), greedy[prompt:])
        assert not library().deepj_hip_token_plan_failed(plan_of(m))
    finally:
        m.close()


def test_ties_and_no_numbers_are_chosen_as_by_the_launches():
    """Equal logits: the lowest index, across tiles and workgroups; a NaN logit above everything; the two zeros are equal."""
    m = model(False, 1500, 40, 256, 8, 1, 300, 1)
    try:
        ids = ref.JavaRandom(1).ints(6, 1500)
        for blm in (np.zeros(1500), np.where(np.arange(1500) % 700 == 699, 3.0, 0.0), np.where(np.arange(1500) == 1234, np.nan, 0.0)):
            tied = LlamaModel(m.cfg, None)
            tied.setTokenGroups(1)
            for name, (r, c) in zip(parameter_names(m.cfg), parameter_shapes(m.cfg)):
                w = np.zeros((r, c), np.float32) if name == "wlm" else np.full((r, c), 0.01, np.float32)
                tied.setWeight(name, blm.astype(np.float32).reshape(1, -1) if name == "blm" else w)
            tied.finalize()
            assert plan_of(tied)
            a = TextGenerator.generate(tied, ids, 8, top_k=1)
            b = TextGenerator.generate(tied, ids, 8, top_k=1, use_graph=False)
            assert np.array_equal(a, b)
            assert np.all(a[6:] == (1234 if np.isnan(blm).any() else int(np.argmax(blm))))
            tied.close()
    finally:
        m.close()


@pytest.mark.parametrize("groups", [1, 8])
def test_a_run_that_cannot_finish_is_done_by_launches(groups):
    """A wait that is given up at once: the run leaves without a token, and tokens, logits, prompts and samples behind it are those
    of the launches."""
    lib = library()
    ids = ref.JavaRandom(9).ints(40, 300)
    good = model(False, 300, 80, 256, 8, 2, 300, -1)
    assert plan_of(good) == 0

    def fresh():
        m = model(False, 300, 80, 256, 8, 2, 300, groups)
        lib.deepj_hip_token_plan_set_polls(plan_of(m), 0)
        return m
    try:
        full = good.forward(ids)
        m = fresh()
        assert np.array_equal(TextGenerator.generate(m, ids[:20], 20, top_k=1), TextGenerator.generate(good, ids[:20], 20, top_k=1))
        assert plan_of(m) == 0                                       # (dropped)
        m.close()
        m = fresh()
        assert np.array_equal(TextGenerator.generate(m, ids[:20], 20, 0.8, 6, 4), TextGenerator.generate(good, ids[:20], 20, 0.8, 6, 4))
        m.close()
        m = fresh()
        assert np.array_equal(TextGenerator.generate(m, ids[:20], 6, 0.8, 0, 4), TextGenerator.generate(good, ids[:20], 6, 0.8, 0, 4))
        m.close()
        m = fresh()
        m.reset()
        m.prefill(ids[:20], choose_next=False)
        for t in range(20, 24):
            m.step(int(ids[t]))
            assert float(np.max(np.abs(m.lastLogits() - full[t]))) <= 2e-4, t
        m.close()
        m = fresh()                                                  # a step and a run whose results nobody reads before the next
        for x in (m, good):
            x.reset()
            x.prefill(ids[:20], choose_next=False)
            x.step(int(ids[20]))
            x.prefill(ids[21:30])
        lib.deepj_hip_token_plan_set_polls(plan_of(m), 0) if plan_of(m) else None
        for x in (m, good):
            x.decode(9)
            x.decode(4)
            x.prefill(ids[30:36])
            x.decode(3)
        assert np.array_equal(m.tokens(), good.tokens())
        assert float(np.max(np.abs(m.lastLogits() - good.lastLogits()))) <= 2e-4
        m.close()
    finally:
        good.close()


@pytest.mark.parametrize("gpt,groups", [(False, 1), (True, 8)])
def test_a_step_leaves_the_state_that_launches_leave(gpt, groups):
    """Steps in front of prompts whose tokens go on as runs and as launches, with and without tokens generated before them."""
    ids = ref.JavaRandom(3).ints(30, 500)
    got = []
    for g in (groups, -1):
        m = model(gpt, 500, 90, 256, 8, 2, 300, g)
        try:
            m.prefill(ids[:5], choose_next=False)
            for t in range(5, 8):
                m.step(int(ids[t]))
            m.prefill(ids[8:10])
            m.decode(6)
            m.step(int(ids[10]))
            m.step(int(ids[11]))
            m.prefill(ids[12:13])
            m.decode(3, use_graph=False)
            m.step(int(ids[13]))
            m.prefill(ids[14:20])
            m.decode(4)
            m.step(int(ids[20]))
            got.append((m.tokens(), m.lastLogits()))
        finally:
            m.close()
    assert np.array_equal(got[0][0], got[1][0]) and len(got[0][0]) == 16
    assert float(np.max(np.abs(got[0][1] - got[1][1]))) <= 2e-4


def test_a_plan_whose_buffer_has_gone_is_refused():
    """Its buffers are looked up again once some buffer has been released: runs go on where another model's have gone, and end where the
    plan's own first one (the embedding) has."""
    lib = library()
    other = model(False, 300, 40, 64, 2, 1, 50, 1)
    base = models._next_id_base[0]
    m = model(False, 300, 40, 256, 8, 1, 300, 1)
    try:
        assert parameter_names(m.cfg)[0] == "emb"
        m.prefill(ref.JavaRandom(1).ints(4, 300))
        other.close()
        m.decode(2)
        m.step(7)
        assert len(m.tokens()) == 3
        lib.deepj_hip_release(np.array([base], dtype=np.int32).ctypes.data, 1)
        assert lib.deepj_hip_token_plan_run(plan_of(m), 1, 1) != 0 and b"released" in lib.deepj_hip_last_error()
        assert lib.deepj_hip_token_plan_step(plan_of(m), 7, 1, 3) != 0 and b"released" in lib.deepj_hip_last_error()
    finally:
        m.close()


def test_plans_are_refused_with_a_reason_or_not_made():
    lib = library()
    m = model(False, 300, 40, 256, 8, 1, 300, 1)
    try:
        plan = plan_of(m)
        assert lib.deepj_hip_token_plan_run(plan, 0, 1) != 0 and b"step count" in lib.deepj_hip_last_error()
        assert lib.deepj_hip_token_plan_run(plan, 2, 0) != 0
        assert lib.deepj_hip_token_plan_run(plan, 1, 2) != 0 and b"choose" in lib.deepj_hip_last_error()
        assert lib.deepj_hip_token_plan_run(plan + 1000, 1, 1) != 0 and b"unknown plan" in lib.deepj_hip_last_error()
        assert lib.deepj_hip_token_plan_set_polls(plan, -1) != 0
        assert lib.deepj_hip_token_plan_step(plan, 40, 1, 0) != 0 and b"context window" in lib.deepj_hip_last_error()
        assert lib.deepj_hip_token_plan_step(plan, -1, 1, 0) != 0
        assert lib.deepj_hip_token_plan_step(plan + 1000, 0, 1, 0) != 0 and b"unknown plan" in lib.deepj_hip_last_error()
    finally:
        m.close()
    assert lib.deepj_hip_token_plan_run(plan, 1, 1) != 0             # gone with its model
    for args in ((300, 40, 256, 2, 1, 300, 8),):                     # two heads for eight groups: launches, not an error
        m = model(False, *args)
        try:
            assert plan_of(m) == 0
            ids = ref.JavaRandom(2).ints(9, 300)
            assert np.array_equal(TextGenerator.generate(m, ids, 9, top_k=1), TextGenerator.generate(m, ids, 9, top_k=1, use_graph=False))
        finally:
            m.close()
    m = LlamaModel(LlamaConfig(64, 16, 64, 2, 1, 96), 1)
    try:
        with pytest.raises(RuntimeError, match="after finalize"):
            m.setTokenGroups(1)
    finally:
        m.close()
    m = LlamaModel(LlamaConfig(64, 16, 64, 2, 1, 96), None)
    with pytest.raises(ValueError, match="token groups must be"):
        m.setTokenGroups(9)
    m.close()


@pytest.mark.parametrize("gpt", [False, True])
@pytest.mark.parametrize("d,heads,groups", [(256, 8, 1), (512, 4, 4), (2112, 33, 8)])
def test_a_first_position_takes_nothing_from_the_rows_an_earlier_sequence_left(gpt, d, heads, groups):
    """A step at position 0 over cache rows that hold no numbers (a sequence with a NaN embedding left them in every block): the
    logits are those of the token alone.  Rows of one and of two sets of values a thread."""
    def with_nan(a):
        a = a.copy()
        a[5] = np.nan
        return a
    m = model(gpt, 300, 40, d, heads, 2, 600, groups, emb=with_nan)
    try:
        assert plan_of(m)
        alone = m.forward([7, 11])
        assert np.isfinite(alone).all()
        for _ in range(2):
            m.reset()
            m.step(5)
            m.step(5)
            assert np.isnan(m.lastLogits()).all()
            m.reset()
            for t, token in enumerate((7, 11)):
                m.step(token)
                assert float(np.max(np.abs(m.lastLogits() - alone[t]))) <= 2e-4, t
    finally:
        m.close()


@pytest.mark.parametrize("gpt,d,heads,groups", [(False, 256, 8, 1), (False, 2112, 33, 8), (True, 256, 8, 1), (True, 768, 12, 8), (True, 2112, 33, 8)])
def test_rows_whose_squares_overflow_are_divided_as_by_the_launches(gpt, d, heads, groups):
    """Finite rows of 1e25: their root mean square (deviation) is infinite, the quotients zero, in every norm of every block."""
    def huge(a):
        a = a.copy()
        a[5] = np.where(np.arange(a.shape[1]) % 2, np.float32(1e25), np.float32(-1e25))
        return a
    got = []
    for g in (groups, -1):
        m = model(gpt, 300, 40, d, heads, 2, 600, g, emb=huge)
        try:
            assert bool(plan_of(m)) == (g > 0)
            m.prefill([3, 4], choose_next=False)
            m.step(5)
            got.append(m.lastLogits())
        finally:
            m.close()
    assert np.isfinite(got[1]).all()
    assert float(np.max(np.abs(got[0] - got[1]))) <= 2e-4


@pytest.mark.parametrize("d,heads,groups", [(256, 8, 1), (2048, 16, 8)])
def test_sums_that_overflow_stay_infinite_behind_the_division(d, heads, groups):
    """Logits whose sums pass the largest float, each of one sign throughout: infinite ones of that sign, as the launches give."""
    def signs(a):
        return np.where(np.arange(a.shape[1]) % 2, np.float32(1), np.float32(-1)) * np.where(np.arange(a.shape[1]) % 3, np.float32(1e4), np.float32(1)) * np.ones_like(a)
    got = []
    for g in (groups, -1):
        m = model(False, 300, 40, d, heads, 2, 600, g, emb=lambda a: 1.0 + np.abs(a), gf=lambda a: np.full_like(a, 1e34), wlm=signs,
                 L1__wd=lambda a: 0 * a, L1__bd=lambda a: 0 * a, L0__wd=lambda a: 0 * a, L0__bd=lambda a: 0 * a, L0__wo=lambda a: 0 * a, L1__wo=lambda a: 0 * a)
        try:
            m.prefill([3, 4], choose_next=False)
            m.step(5)
            got.append(m.lastLogits())
        finally:
            m.close()
    assert np.isinf(got[1]).any() and np.isfinite(got[1]).any()
    assert np.array_equal(np.isinf(got[0]), np.isinf(got[1])) and np.array_equal(np.sign(got[0]), np.sign(got[1]))
    both = np.isfinite(got[1])
    assert float(np.max(np.abs(got[0][both] / got[1][both] - 1))) <= 1e-5


class RawPlan:
    """A plan over zeroed buffers of the test's own: one Llama block on one group, heads of 32."""
    def __init__(self, base, shape=None, room=True):
        lib = library()
        self.shape = s = shape or dict(vocab=64, max_seq=40, d=64, heads=2, dff=64)
        d, f, v, n = s["d"], s["dff"], s["vocab"], s["max_seq"]
        q8 = lib.deepj_hip_q8_floats
        sizes = dict(emb=v * d, gf=d, wlm=q8(d, v), blm=v, cos=n * 16, sin=n * 16, kc=n * d, vc=n * d, state=4, tokens=n, logits=v, x=d,
                     g1=d, g2=d, wqkv=q8(d, 3 * d), wo=q8(d, d), wgu=q8(d, 2 * f), bg=f, bu=f, wd=q8(f, d), bd=d)
        self.id = {name: base + i for i, name in enumerate(sizes)}
        self.sizes = sizes
        ids, counts = (np.array(list(a), dtype=np.int32) for a in (self.id.values(), sizes.values()))
        assert lib.deepj_hip_alloc_buffers(ids.ctypes.data, counts.ctypes.data, len(ids)) == 0
        fills = Stream()
        for name in sizes:
            fills.emit(op.OP_FILL, self.id[name], 0, sizes[name])
        HipNative.nativeFlushOps(fills.array(), len(fills.array()))
        self.plan = 0
        self.make(room)

    def make(self, room=True):
        b, s = self.id, self.shape
        words = np.array([0, s["vocab"], s["max_seq"], s["d"], s["heads"], 1, s["dff"], 1, b["emb"], -1, b["gf"], -1, b["wlm"], b["blm"], b["cos"], b["sin"],
                          b["kc"], b["vc"], b["state"], b["tokens"], b["logits"], b["x"],
                          b["g1"], -1, b["g2"], -1, b["wqkv"], b["wo"], b["wgu"], b["bg"], b["bu"], b["wd"], b["bd"]], dtype=np.int32)
        plan = C.c_int32()
        assert library().deepj_hip_token_plan_create(words.ctypes.data_as(C.c_void_p), len(words), C.byref(plan)) == 0 and bool(plan.value) == room
        self.plan = plan.value

    def state(self):
        out = np.empty(4, dtype=np.int32)
        assert library().deepj_hip_download(self.id["state"], out.ctypes.data, 4) == 0
        return out.tolist()

    def close(self):
        lib = library()
        if self.plan:
            lib.deepj_hip_token_plan_destroy(self.plan)
        ids = np.array(list(self.id.values()), dtype=np.int32)
        lib.deepj_hip_release(ids.ctypes.data, len(ids))


@pytest.fixture
def raw():
    HipNative.init(0)
    p = RawPlan(1 << 28)
    yield p
    p.close()


def test_runs_behind_one_that_gave_up_do_nothing(raw):
    """Each would wait as long for the same workgroups.  The state stays behind the last whole token."""
    lib = library()
    assert lib.deepj_hip_token_plan_run(raw.plan, 2, 1) == 0
    lib.deepj_hip_token_plan_set_polls(raw.plan, 0)
    assert lib.deepj_hip_token_plan_run(raw.plan, 3, 1) == 0
    lib.deepj_hip_token_plan_set_polls(raw.plan, 1 << 21)
    assert lib.deepj_hip_token_plan_run(raw.plan, 3, 1) == 0          # (on its way before the host can know)
    assert raw.state() == [2, 0, 2, 0] and lib.deepj_hip_token_plan_failed(raw.plan)
    assert lib.deepj_hip_token_plan_run(raw.plan, 3, 1) == 0
    assert lib.deepj_hip_token_plan_step(raw.plan, 7, 1, 3) == 0
    assert raw.state() == [2, 0, 2, 0]


def test_calls_behind_a_run_wait_for_nothing():
    """Tokens one at a time, forced ones and a prompt, behind work that takes the device far longer than their calls the host."""
    lib = library()
    m = model(False, 300, 80, 256, 8, 2, 300, 1)
    big, size = np.array([1 << 28], dtype=np.int32), np.array([1 << 28], dtype=np.int32)
    assert lib.deepj_hip_alloc_buffers(big.ctypes.data, size.ctypes.data, 1) == 0
    try:
        ids = ref.JavaRandom(3).ints(40, 300)
        fills = Stream()
        for _ in range(400):
            fills.emit(op.OP_FILL, int(big[0]), 0, int(size[0]))
        fills = fills.array()

        def calls():
            m.reset()
            m.prefill(ids[:20])
            for _ in range(4):
                m.decode(1)
            m.step(int(ids[20]))
            m.step(int(ids[21]))
            m.prefill(ids[22:30])
            m.decode(2)
        calls()
        tokens = m.tokens()
        start = time.perf_counter()
        HipNative.nativeFlushOps(fills, len(fills))
        calls()
        called = time.perf_counter() - start
        assert np.array_equal(m.tokens(), tokens) and len(tokens) == 8
        assert called < 0.5 * (time.perf_counter() - start), called
    finally:
        lib.deepj_hip_release(big.ctypes.data, 1)
        m.close()


@pytest.mark.parametrize("gpt,groups", [(False, 1), (True, 8), (False, 4)])
def test_everything_behind_a_run_that_gave_up_is_done_again(gpt, groups):
    """Runs, steps and prompts whose results nobody reads in between, with the wait that is given up at each of them: tokens and
    logits are those of the launches."""
    lib = library()
    ids = ref.JavaRandom(9).ints(40, 300)
    calls = [lambda m: m.decode(3), lambda m: m.decode(1), lambda m: m.step(int(ids[5])), lambda m: m.step(int(ids[6])),
             lambda m: m.prefill(ids[7:9]), lambda m: m.decode(4), lambda m: m.prefill(ids[9:14], choose_next=False),
             lambda m: m.step(int(ids[14])), lambda m: m.prefill(ids[15:33]), lambda m: m.decode(2), lambda m: m.decode(5)]

    def results(m, ends, at=None):
        m.reset()
        m.prefill(ids[:5])
        for i, call in enumerate(calls[:ends]):
            if i == at:
                lib.deepj_hip_token_plan_set_polls(plan_of(m), 0)
            call(m)
        return (m.lastLogits(), m.tokens()) if ends % 2 else (m.tokens(), m.lastLogits())[::-1]
    good = model(gpt, 300, 90, 256, 8, 2, 600, -1)
    try:
        for ends in (1, 4, 8, 11):
            logits, tokens = results(good, ends)
            for at in range(ends):
                m = model(gpt, 300, 90, 256, 8, 2, 600, groups)
                try:
                    got = results(m, ends, at)
                    late = all(i in (4, 6, 8) for i in range(at, ends))       # (no run behind it)
                    assert bool(plan_of(m)) == late, (ends, at)
                    assert np.array_equal(got[1], tokens), (ends, at)
                    assert float(np.max(np.abs(got[0] - logits))) <= 2e-4, (ends, at)
                finally:
                    m.close()
    finally:
        good.close()


def test_rows_of_a_prompt_behind_a_run_that_gave_up():
    """Every row's logits of a prompt whose cache the run left short."""
    m, good = (model(False, 300, 90, 256, 8, 2, 300, g) for g in (1, -1))
    try:
        ids = ref.JavaRandom(4).ints(30, 300)
        library().deepj_hip_token_plan_set_polls(plan_of(m), 0)
        got = []
        for x in (m, good):
            x.prefill(ids[:9])
            x.decode(4)
            out = np.empty((17, 300), dtype=np.float32)
            chunk = np.ascontiguousarray(ids[9:26])
            assert library().deepj_runner_prefill(x._h, chunk.ctypes.data_as(C.POINTER(C.c_int32)), 17, out.ctypes.data, 1) == 0
            x.decode(3)
            got.append((out, x.tokens()))
        assert float(np.max(np.abs(got[0][0] - got[1][0]))) <= 2e-4 and np.array_equal(got[0][1], got[1][1])
    finally:
        m.close()
        good.close()


class limited:
    """Device memory that the library may take beyond what its buffers hold now, in bytes."""

    def __init__(self, more):
        self.more = more

    def __enter__(self):
        library().deepj_hip_trim()
        assert library().deepj_hip_limit_memory(C.c_int64(self.more)) == 0

    def __exit__(self, *exc):
        library().deepj_hip_limit_memory(C.c_int64(-1))


def test_a_model_that_fits_without_a_plan_loads_without_one():
    """Memory for the weights, their fp16 copies and the prompt's buffers, and not for the plan."""
    shape = (False, 3000, 512, 1024, 16, 2, 2816)
    before = HipNative.poolStats()["live_bytes"]
    plain = model(*shape, -1)                                        # (the workspaces are at their sizes behind it)
    need, copies = HipNative.poolStats()["live_bytes"] - before, plain.preparedBytes()
    plain.close()
    assert copies > 0
    with limited(need):
        m = model(*shape, 8)
        try:
            assert plan_of(m) == 0 and m.preparedBytes() == copies
            ids = ref.JavaRandom(2).ints(30, 3000)
            assert np.array_equal(TextGenerator.generate(m, ids, 9, top_k=1), TextGenerator.generate(m, ids, 9, top_k=1, use_graph=False))
        finally:
            m.close()
    m = model(*shape, 8)
    assert plan_of(m) and m.preparedBytes() == copies
    m.close()


def test_a_plan_gives_its_memory_back_where_other_memory_is_short():
    """For a buffer that would not fit beside it; tokens behind it, and those of runs that nobody had looked at, are right.  Another
    plan is no reason."""
    lib = library()
    shape = (False, 3000, 200, 1024, 16, 2, 2816)
    ids = ref.JavaRandom(2).ints(30, 3000)
    m = model(*shape, 8)
    one, size = np.array([1 << 28], dtype=np.int32), np.array([1 << 18], dtype=np.int32)
    try:
        exp = TextGenerator.generate(m, ids, 12, top_k=1, use_graph=False)[30:]
        m.reset()
        m.prefill(ids)
        m.decode(5)
        plan = plan_of(m)
        before = HipNative.poolStats()["live_bytes"]
        raw = RawPlan(1 << 27)
        raw_bytes = HipNative.poolStats()["live_bytes"] - before
        raw.close()
        with limited(raw_bytes - 1024):                               # (all of it but its plan)
            raw = RawPlan(1 << 27, room=False)
            assert plan_of(m) == plan
            raw.close()
        with limited(0):
            assert lib.deepj_hip_alloc_buffers(one.ctypes.data, size.ctypes.data, 1) == 0
        assert plan_of(m) == 0
        assert lib.deepj_hip_token_plan_run(plan, 1, 1) != 0 and b"given back" in lib.deepj_hip_last_error()
        m.decode(4)
        m.decode(2)
        assert np.array_equal(m.tokens(), exp)
        assert np.array_equal(TextGenerator.generate(m, ids, 12, top_k=1)[30:], exp)
        with limited(0):                                              # with nothing left to give back
            size[0] = 1 << 28
            one[0] += 1
            assert lib.deepj_hip_alloc_buffers(one.ctypes.data, size.ctypes.data, 1) != 0 and b"Failed to allocate" in lib.deepj_hip_last_error()
    finally:
        lib.deepj_hip_release(np.array([1 << 28], dtype=np.int32).ctypes.data, 1)
        m.close()

def test_a_run_of_a_plan_that_has_gone_marks_no_other(raw):
    """A run that gives up behind its plan's end, with another plan made meanwhile: the other one has not failed."""
    lib = library()
    big, size = np.array([(1 << 28) + 1000], dtype=np.int32), np.array([1 << 26], dtype=np.int32)
    assert lib.deepj_hip_alloc_buffers(big.ctypes.data, size.ctypes.data, 1) == 0
    try:
        fills = Stream()
        for _ in range(400):
            fills.emit(op.OP_FILL, int(big[0]), 0, int(size[0]))
        HipNative.nativeFlushOps(fills.array(), len(fills.array()))       # (some 20 ms that the run stands behind)
        lib.deepj_hip_token_plan_set_polls(raw.plan, 0)
        assert lib.deepj_hip_token_plan_run(raw.plan, 3, 1) == 0
        lib.deepj_hip_token_plan_destroy(raw.plan)
        raw.make()
        assert lib.deepj_hip_synchronize() == 0
        assert not lib.deepj_hip_token_plan_failed(raw.plan)
        assert lib.deepj_hip_token_plan_run(raw.plan, 3, 1) == 0 and raw.state()[0] == 3
    finally:
        lib.deepj_hip_release(big.ctypes.data, 1)

def test_a_plan_over_a_buffer_that_was_made_again_is_refused(raw):
    """Also where the new buffer of that id lies where the old one did: the plan's copies are of what the old one held."""
    lib = library()
    assert lib.deepj_hip_token_plan_run(raw.plan, 2, 1) == 0 and raw.state()[0] == 2
    one, size = np.array([raw.id["wo"]], dtype=np.int32), np.array([raw.sizes["wo"]], dtype=np.int32)
    assert lib.deepj_hip_release(one.ctypes.data, 1) == 0
    assert lib.deepj_hip_alloc_buffers(one.ctypes.data, size.ctypes.data, 1) == 0
    assert lib.deepj_hip_token_plan_run(raw.plan, 1, 1) != 0 and b"released" in lib.deepj_hip_last_error()


@pytest.mark.parametrize("gpt,groups", [(False, 1), (True, 8)])
def test_a_run_of_more_tokens_than_a_launch_takes(gpt, groups):
    """300 and 600 tokens, in launches of 256, against the launches of a token."""
    m = model(gpt, 300, 700, 256, 8, 2, 600, groups)
    try:
        ids = ref.JavaRandom(6).ints(20, 300)
        exp = TextGenerator.generate(m, ids, 601, top_k=1, use_graph=False)
        assert np.array_equal(TextGenerator.generate(m, ids, 301, top_k=1), exp[:321])
        assert np.array_equal(TextGenerator.generate(m, ids, 601, top_k=1), exp)
        assert plan_of(m)
    finally:
        m.close()


@pytest.mark.parametrize("gpt,groups", [(False, 1), (True, 8)])
def test_tags_start_over(gpt, groups):
    """The words' numbers at the end of 32 bits: a token has 24 here, a run one more.  Runs that just fit, just do not, and steps."""
    lib = library()
    ids = ref.JavaRandom(6).ints(20, 300)
    m = model(gpt, 300, 90, 256, 8, 2, 600, groups)
    try:
        exp = TextGenerator.generate(m, ids, 14, top_k=1, use_graph=False)[20:]
    finally:
        m.close()
    for left in (0, 1, 24, 25, 26, 48, 49, 50, 73, 74, 200):
        m = model(gpt, 300, 90, 256, 8, 2, 600, groups)
        try:
            plan = plan_of(m)
            m.prefill(ids)
            m.decode(3)
            assert lib.deepj_hip_token_plan_set_tag(plan, C.c_uint32(0xffffffff - left)) == 0
            m.decode(2)
            m.decode(1)
            m.decode(3)
            assert lib.deepj_hip_token_plan_set_tag(plan, C.c_uint32(1)) != 0 and b"exchange block" in lib.deepj_hip_last_error()
            m.decode(4)
            assert np.array_equal(m.tokens(), exp) and plan_of(m), left
            m.step(5)
            logits = m.lastLogits()
            m.reset()
            m.prefill(np.concatenate([ids, exp[:13]]), choose_next=False)
            m.step(5)
            assert np.array_equal(m.lastLogits().view(np.int32), logits.view(np.int32)) or np.max(np.abs(m.lastLogits() - logits)) <= 2e-4
        finally:
            m.close()


@pytest.mark.parametrize("gpt,d,heads,dff,groups", [(False, 64, 2, 50, 1), (False, 256, 8, 600, 1), (True, 256, 8, 600, 1), (False, 320, 10, 1000, 4), (True, 768, 12, 3072, 8), (False, 2112, 33, 5000, 8)])
def test_words_through_memory_are_the_words_of_a_shared_l2(gpt, d, heads, dff, groups):
    """Groups whose workgroups do not share an XCD: the same bits."""
    m = model(gpt, 1003, 200, d, heads, 2, dff, groups)
    try:
        ids = ref.JavaRandom(6).ints(100, 1003)
        got = []
        for far in (0, 1, 0):
            assert library().deepj_hip_token_plan_set_far(plan_of(m), far) == 0
            tokens = TextGenerator.generate(m, ids, 40, top_k=1)
            m.step(7)
            got.append((tokens, m.lastLogits()))
        for tokens, logits in got[1:]:
            assert np.array_equal(tokens, got[0][0]) and np.array_equal(logits.view(np.int32), got[0][1].view(np.int32))
        assert plan_of(m)
    finally:
        m.close()


@pytest.mark.parametrize("gpt,groups", [(False, 1), (True, 8)])
def test_a_run_that_gives_up_somewhere_is_done_again(gpt, groups):
    """Waits of a few loads.  Whether one ends a run, and in front of which token (the next test's runs end behind some), is the device's
    choice, and what comes out is not."""
    ids = ref.JavaRandom(9).ints(20, 300)
    good = model(gpt, 300, 90, 256, 8, 2, 600, -1)
    try:
        exp = TextGenerator.generate(good, ids, 40, top_k=1)[20:]
        good.step(3)
        logits = good.lastLogits()
    finally:
        good.close()
    for polls in (1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 64):
        m = model(gpt, 300, 90, 256, 8, 2, 600, groups)
        try:
            library().deepj_hip_token_plan_set_polls(plan_of(m), polls)
            m.prefill(ids)
            m.decode(30)
            m.decode(9)
            m.step(3)
            assert float(np.max(np.abs(m.lastLogits() - logits))) <= 2e-4, polls
            assert np.array_equal(m.tokens(), exp), polls
        finally:
            m.close()


def test_a_run_that_gives_up_leaves_the_state_behind_a_whole_token():
    """What the plan's caller finds.  Over 390000 positions two of a group's 32 workgroups, which three heads leave without keys, wait
    far longer for the others in every token than for their start, so that a bound near that wait ends runs behind some of their tokens:
    sought by halves, then tried until one did."""
    HipNative.init(0)
    lib, start, asked = library(), 390000, 30
    raw = RawPlan(1 << 28, dict(vocab=64, max_seq=400000, d=96, heads=3, dff=64))

    def reached(polls):
        lib.deepj_hip_token_plan_destroy(raw.plan)
        raw.make()
        lib.deepj_hip_token_plan_set_polls(raw.plan, polls)
        lib.deepj_hip_upload(raw.id["state"], np.array([start, 0, 0, 0], dtype=np.int32).ctypes.data, 4)
        lib.deepj_hip_upload(raw.id["tokens"], np.full(asked + 1, -1, dtype=np.int32).ctypes.data, asked + 1)
        assert lib.deepj_hip_token_plan_run(raw.plan, asked, 1) == 0
        pos, token, generated, _ = raw.state()
        tokens = np.empty(asked + 1, dtype=np.int32)
        lib.deepj_hip_download(raw.id["tokens"], tokens.ctypes.data, asked + 1)
        assert 0 <= generated <= asked and pos == start + generated and token == 0
        assert np.all(tokens[:generated] == 0) and np.all(tokens[generated:] == -1)
        assert generated == asked or lib.deepj_hip_token_plan_failed(raw.plan)
        return generated
    try:
        assert reached(1 << 21) == asked and reached(0) == 0
        some, low, high = [], 1, 1 << 16
        while high > low * 1.01 + 1:
            polls = int((low * high) ** 0.5)
            some.append(reached(polls))
            low, high = (low, polls) if some[-1] == asked else (polls, high)
        while not any(0 < n < asked for n in some) and len(some) < 300:
            some.append(reached(low + len(some) % 64))
        if not any(0 < n < asked for n in some):
            pytest.skip("no run ended inside its tokens")
    finally:
        raw.close()


@pytest.mark.parametrize("warms_up", [True, False])
def test_loading_a_model_runs_a_token_of_its_plan(warms_up, monkeypatch):
    """The first launch of the kernel is the loading's, not the first request's, unless warming up is switched off.  (A plan no run
    has been launched of takes any number for its first words.)"""
    if not warms_up:
        monkeypatch.setenv("DEEPJ_HIP_WARMUP", "0")
    m = model(False, 300, 40, 256, 8, 2, 600, 1)
    try:
        assert (library().deepj_hip_token_plan_set_tag(plan_of(m), C.c_uint32(1)) != 0) == warms_up
        assert len(m.tokens()) == 0
        ids = ref.JavaRandom(6).ints(5, 300)
        assert np.array_equal(TextGenerator.generate(m, ids, 9, top_k=1), TextGenerator.generate(m, ids, 9, top_k=1, use_graph=False))
    finally:
        m.close()
