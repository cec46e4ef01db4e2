"""The work this library is measured on: what a program that uses it has it do, through its public entry points, from
one token of a small model to a prompt of 2048 rows.

Two kinds of program use the library.  One holds a decoder model (deepj_amd.models) and generates, scores or steps
through text; its weights are Q8 on the device and its results are token ids or logits on the host.  The other records
tensor operations (deepj_amd.tensor over HipBackend) or fused operations (deepj_amd.fused) of its own: an unmodified
layer library run through the backend, a training step, a feed-forward block on Q8 weights.

listed() names twelve cases, draw() gives more of the same ranges, prepare() makes what such a program holds before the
call (weights, prompts, tensors; all from the seed), run() is one pass of it.  Weights are N(0, 1 / d): activations,
attention scores and logits then have the spread they have in trained models.
"""
from __future__ import annotations

import itertools
import math

import numpy as np
import torch

from deepj_amd import (DeepSeekConfig, DeepSeekModel, GPTConfig, GPTModel, HipBackend, HipNative, LlamaConfig, LlamaModel,
                       Tensor, TextGenerator, parameter_names, parameter_shapes)
from deepj_amd.fused import DeviceBuffers, Stream

# ── the cases ────────────────────────────────────────────────────────────────


def listed():
    return [
        # A small model answering a short prompt, greedily: nothing but launches and the latency of each.
        dict(name="greedy_small", kind="greedy", family="llama", vocab=256, max_seq=256, d=256, heads=8, layers=4, dff=688,
             q_rank=0, kv_rank=0, prompt=16, new=48),
        # The headline workload: batch-1 greedy decode of a 1 B parameter Llama behind a 512-token prompt.
        dict(name="greedy_llama", kind="greedy", family="llama", vocab=32000, max_seq=2048, d=2048, heads=32, layers=16, dff=5632,
             q_rank=0, kv_rank=0, prompt=512, new=64),
        # The same for the DeepSeek model with the latent KV cache (chosen where memory is short): every token expands the
        # cached latent rows again.
        dict(name="greedy_latent", kind="greedy", family="latent", vocab=32000, max_seq=1024, d=2048, heads=16, layers=4, dff=5632,
             q_rank=1024, kv_rank=512, prompt=300, new=24),
        # Sampled generation (temperature, top-k) with a large vocabulary: the text generator as chat programs use it.
        dict(name="sampled_gpt", kind="sampled", family="gpt", vocab=50257, max_seq=1024, d=768, heads=12, layers=12, dff=3072,
             q_rank=0, kv_rank=0, prompt=90, new=40, temperature=0.8, top_k=40),
        # A conversation: each turn appends some tokens of a user's to the cached context and generates a reply.
        dict(name="turns_llama", kind="turns", family="llama", vocab=32000, max_seq=2048, d=2048, heads=32, layers=4, dff=5632,
             q_rank=0, kv_rank=0, prompt=611, turn=29, turns=3, new=16),
        # Tokens chosen by the caller (constrained decoding, an outside sampler): every step hands back its logits.
        dict(name="steps_llama", kind="steps", family="llama", vocab=8192, max_seq=512, d=1024, heads=16, layers=8, dff=2752,
             q_rank=0, kv_rank=0, prompt=75, new=32),
        # A long prompt through wide layers: the largest matrix products.
        dict(name="prompt_wide", kind="prompt", family="llama", vocab=32000, max_seq=2048, d=4096, heads=32, layers=4, dff=11008,
             q_rank=0, kv_rank=0, prompt=2048),
        # Scoring a text: logits of every row of the sequence (perplexity, ranking of answers).
        dict(name="score_gpt", kind="score", family="gpt", vocab=50257, max_seq=1024, d=768, heads=12, layers=12, dff=3072,
             q_rank=0, kv_rank=0, prompt=400),
        # An attention layer of an unmodified layer library: heads split, masked and merged on the host, every product and
        # soft-max a tensor operation of its own.
        dict(name="layer_attention", kind="attention", rows=64, d=256, heads=8),
        # A norm and a gated feed-forward layer composed of tensor operations on fp32 weights.
        dict(name="layer_ffn", kind="ffn", rows=500, d=1024, dff=2752),
        # Training steps of a small language model: forward, loss, backward, AdamW, then the parameters for a checkpoint.
        dict(name="train_small", kind="train", rows=256, d=192, dff=768, vocab=1003, steps=6),
        # A gated feed-forward block on Q8 weights as fused operations, for a batch of rows.
        dict(name="q8_ffn", kind="q8_ffn", rows=64, d=4096, dff=11008, prepared=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _drawn_model(rng, families, max_params):
    """A model's dimensions: heads of 32, 64 or 128, a feed-forward width between two and four times the model's, an
    ordinary or an odd vocabulary."""
    family = rng.choice(families)
    while True:
        hd = rng.choice([32, 64, 64, 128])
        d = hd * max(1, round(_log_int(rng, 128, 2560) / hd))
        layers = _log_int(rng, 2, 16)
        dff = 8 * round(rng.uniform(2.0, 4.0) * d / 8)
        vocab = _log_int(rng, 256, 50257)
        case = dict(family=family, vocab=vocab, max_seq=1024, d=d, heads=d // hd, layers=layers, dff=dff, q_rank=0, kv_rank=0)
        if family in ("deepseek", "latent"):
            case.update(q_rank=max(8, d // 2), kv_rank=max(8, d // 4))
        if sum(r * c for r, c in parameter_shapes(_config(case))) <= max_params:
            return case


def draw(rng):
    kind = rng.choice(["greedy", "greedy", "sampled", "turns", "steps", "prompt", "score", "attention", "ffn", "train", "q8_ffn", "q8_ffn"])
    if kind == "greedy":
        m = _drawn_model(rng, ["llama", "gpt", "deepseek", "latent"], 2.5e8)
        return dict(m, kind=kind, prompt=_log_int(rng, 4, 700), new=_log_int(rng, 12, 40))
    if kind == "sampled":
        m = _drawn_model(rng, ["llama", "gpt"], 2.0e8)
        return dict(m, kind=kind, prompt=_log_int(rng, 4, 500), new=_log_int(rng, 12, 40), temperature=round(rng.uniform(0.5, 1.2), 2),
                    top_k=rng.choice([0, 5, 20, 50, 200]))
    if kind == "turns":
        m = _drawn_model(rng, ["llama", "gpt", "deepseek", "latent"], 2.0e8)
        return dict(m, kind=kind, prompt=_log_int(rng, 20, 700), turn=_log_int(rng, 2, 60), turns=rng.randint(2, 3), new=_log_int(rng, 8, 20))
    if kind == "steps":
        m = _drawn_model(rng, ["llama", "gpt", "deepseek"], 2.0e8)
        return dict(m, kind=kind, prompt=_log_int(rng, 4, 500), new=_log_int(rng, 8, 40))
    if kind == "prompt":
        m = _drawn_model(rng, ["llama", "gpt", "deepseek"], 3.0e8)
        return dict(m, kind=kind, prompt=_log_int(rng, 8, 1024))
    if kind == "score":
        m = _drawn_model(rng, ["llama", "gpt"], 2.0e8)
        return dict(m, kind=kind, prompt=_log_int(rng, 8, 400))
    if kind == "attention":
        hd = rng.choice([32, 64])
        heads = rng.randint(2, 12)
        return dict(kind=kind, rows=_log_int(rng, 8, 160), d=hd * heads, heads=heads)
    if kind == "ffn":
        d = _log_int(rng, 64, 2048)
        return dict(kind=kind, rows=_log_int(rng, 1, 1024), d=d, dff=round(rng.uniform(2.0, 3.5) * d))
    if kind == "train":
        d = 8 * _log_int(rng, 8, 64)
        return dict(kind=kind, rows=_log_int(rng, 16, 512), d=d, dff=4 * d, vocab=_log_int(rng, 64, 4096), steps=rng.randint(2, 6))
    d = 8 * _log_int(rng, 32, 512)
    return dict(kind=kind, rows=_log_int(rng, 1, 1024), d=d, dff=8 * round(rng.uniform(2.0, 3.0) * d / 8), prepared=rng.random() < 0.5)


# ── what a program holds before the call ─────────────────────────────────────


def _gaussians(n, seed, scale):
    """n values of N(0, scale) on the host, made on the GPU from the seed."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(n, generator=gen, device="cuda") * scale).cpu().numpy()


def _config(c):
    args = (c["vocab"], c["max_seq"], c["d"], c["heads"], c["layers"], c["dff"])
    if c["family"] == "gpt":
        return GPTConfig(*args)
    if c["family"] in ("deepseek", "latent"):
        return DeepSeekConfig(*args, c["q_rank"], c["kv_rank"])
    return LlamaConfig(*args)


def _model(c, seed):
    cfg = _config(c)
    if c["family"] == "gpt":
        model = GPTModel(cfg, None)
    elif c["family"] in ("deepseek", "latent"):
        model = DeepSeekModel(cfg, None, latent_cache=c["family"] == "latent")
    else:
        model = LlamaModel(cfg, None)
    shapes = parameter_shapes(cfg)
    # one pool of values, every parameter a stretch of it that begins elsewhere
    pool = _gaussians(max(r * k for r, k in shapes) + (1 << 20), seed, c["d"] ** -0.5)
    starts = np.random.default_rng(seed).integers(0, 1 << 20, len(shapes))
    for name, (r, k), at in zip(parameter_names(cfg), shapes, starts):
        a = pool[at:at + r * k].reshape(r, k)
        leaf = name.split(".")[-1]
        model.setWeight(name, 1.0 + a if leaf in ("g1", "g2", "gf") else a)
    model.finalize()
    return model


_backend = []
_id_bases = itertools.count(1 << 28, 1 << 10)


def _tensors():
    """The tensor backend of this process (one for all: it hands out the buffer ids)."""
    if not _backend:
        _backend.append(HipBackend())
        Tensor.setBackend(_backend[0])


class _Buffers(DeviceBuffers):
    def __init__(self):
        super().__init__(next(_id_bases))

    def __del__(self):
        self.release_all()


def prepare(case, seed):
    kind, rng = case["kind"], np.random.default_rng(seed)
    if kind in ("greedy", "sampled", "turns", "steps", "prompt", "score"):
        state = dict(case, model=_model(case, seed), prompt_ids=rng.integers(0, case["vocab"], case["prompt"]).astype(np.int32), seed=seed)
        if kind == "turns":
            state["turn_ids"] = [rng.integers(0, case["vocab"], case["turn"]).astype(np.int32) for _ in range(case["turns"])]
        if kind == "steps":
            state["chosen"] = [int(t) for t in rng.integers(0, case["vocab"], case["new"])]
        return state

    if kind == "q8_ffn":
        dev, rows, d, dff = _Buffers(), case["rows"], case["d"], case["dff"]
        pool = _gaussians(3 * d * dff, seed, d ** -0.5)
        wgu, wd = dev.alloc(HipNative.q8Floats(d, 2 * dff)), dev.alloc(HipNative.q8Floats(dff, d))
        for k, (dst, r, c, off, step, total) in enumerate(((wgu, d, dff, 0, 2, 2 * dff), (wgu, d, dff, 1, 2, 2 * dff), (wd, dff, d, 0, 1, d))):
            src = dev.upload(pool[k * d * dff:(k + 1) * d * dff])
            Stream().q8_quantize(src, dst, r, c, off, step, total).run()
            dev.release(src)
        if case["prepared"]:
            for w, k, n in ((wgu, d, 2 * dff), (wd, dff, d)):
                Stream().q8_prepare(w, dev.alloc(HipNative.q8PreparedFloats(k, n)), k, n).run()
        x = rng.standard_normal((rows, d)).astype(np.float32)
        gamma = dev.upload((1.0 + 0.1 * rng.standard_normal(d)).astype(np.float32))
        bg, bu, bd = (dev.upload((0.1 * rng.standard_normal(n)).astype(np.float32)) for n in (dff, dff, d))
        xb, hb, ob = dev.alloc(rows * d), dev.alloc(rows * dff), dev.alloc(rows * d)
        stream = (Stream().q8_linear(xb, wgu, hb, rows, d, dff, gamma=gamma, bias=bg, bias2=bu, swiglu=True)
                  .q8_linear(hb, wd, ob, rows, dff, d, bias=bd, residual=xb))
        HipNative.synchronize()
        return dict(case, dev=dev, x=x, xb=xb, ob=ob, stream=stream)

    _tensors()
    rows, d = case["rows"], case["d"]

    def tensor(r, c, scale, mean=0.0):
        return Tensor.from2D(rng.standard_normal((r, c), dtype=np.float32) * np.float32(scale) + np.float32(mean))

    if kind == "attention":
        return dict(case, x=tensor(rows, d, 1.0), weights=[tensor(d, d, d ** -0.5) for _ in range(4)], mask=Tensor.causalMask(rows))
    if kind == "ffn":
        dff = case["dff"]
        return dict(case, x=tensor(rows, d, 1.0), gamma=tensor(1, d, 0.1, 1.0), wg=tensor(d, dff, d ** -0.5), bg=tensor(1, dff, 0.1),
                    wu=tensor(d, dff, d ** -0.5), bu=tensor(1, dff, 0.1), wd=tensor(dff, d, dff ** -0.5), bd=tensor(1, d, 0.1))
    dff, vocab = case["dff"], case["vocab"]
    shapes = {"emb": (vocab, d), "gamma": (1, d), "beta": (1, d), "w1": (d, dff), "b1": (1, dff), "w2": (dff, d), "b2": (1, d),
              "wh": (d, vocab), "bh": (1, vocab)}
    params = {n: tensor(r, c, 0.02 if r == 1 else r ** -0.5 if n != "emb" else 1.0, 1.0 if n == "gamma" else 0.0) for n, (r, c) in shapes.items()}
    moments = {n: (Tensor.zeros(r, c), Tensor.zeros(r, c)) for n, (r, c) in shapes.items()}
    batches = [(rng.integers(0, vocab, rows), rng.integers(0, vocab, rows)) for _ in range(case["steps"])]
    return dict(case, params=params, moments=moments, batches=batches, step=0)


# ── one pass ─────────────────────────────────────────────────────────────────


def _turns(s):
    model, replies = s["model"], []
    model.reset()
    ids = s["prompt_ids"]
    for turn in [None, *s["turn_ids"]]:
        if turn is not None:                     # the reply's last token is not in the cache yet
            ids = np.concatenate([replies[-1][-1:], turn])
        model.prefill(ids)
        model.decode(s["new"] - 1)
        replies.append(model.tokens())           # all tokens generated in this sequence so far
    return replies[-1]


def _steps(s):
    model = s["model"]
    model.reset()
    model.prefill(s["prompt_ids"], choose_next=False)
    out = [model.lastLogits()]
    for token in s["chosen"]:
        model.step(token)
        out.append(model.lastLogits())
    return out


def _attention(s):
    """Multi-head attention as a layer library composes it over tensors: per-head blocks are cut out and put back on the
    host, scores, mask and values are products and sums of their own."""
    rows, heads, hd = s["rows"], s["heads"], s["d"] // s["heads"]
    wq, wk, wv, wo = s["weights"]
    q, k, v = (s["x"].matmul(w).numpy() for w in (wq, wk, wv))
    scores, merged = Tensor(heads * rows, rows), Tensor(rows, s["d"])
    for h in range(heads):
        cols = slice(h * hd, (h + 1) * hd)
        sc = Tensor.from2D(q[:, cols]).matmul(Tensor.from2D(k[:, cols]).transpose())
        scores.data[h * rows:(h + 1) * rows] = sc.multiplyScalarInPlace(hd ** -0.5).add(s["mask"]).numpy()
    probs = scores.softmaxRows().numpy()
    for h in range(heads):
        cols = slice(h * hd, (h + 1) * hd)
        merged.data[:, cols] = Tensor.from2D(probs[h * rows:(h + 1) * rows]).matmul(Tensor.from2D(v[:, cols])).numpy()
    return merged.matmul(wo).numpy()


def _ffn(s):
    """x + down(SiLU(gate(norm(x))) * up(norm(x))), RMSNorm and SiLU composed of their operations."""
    x = s["x"]
    rms = x.multiply(x).meanAlongRows().addScalar(1e-6).sqrt()
    n = x.divideBroadcastCols(rms).multiplyBroadcastRows(s["gamma"])
    gate = n.matmul(s["wg"]).addRowVector(s["bg"])
    up = n.matmul(s["wu"]).addRowVector(s["bu"])
    fused = gate.multiply(gate.sigmoidActivation()).multiply(up)
    return fused.matmul(s["wd"]).addRowVector(s["bd"]).add(x).numpy()


def _train(s):
    """Steps of: token rows, LayerNorm, GELU feed-forward with a residual, vocabulary head; cross entropy, its gradients,
    AdamW on every parameter.  The losses are read at every step, parameters, moments and last gradients at the end."""
    p, d = s["params"], s["d"]
    losses, grads = [], {}
    for ids, targets in s["batches"]:
        x = Tensor.sliceRows(p["emb"], ids, d)
        centred = x.subtractBroadcastCols(x.meanAlongRows())
        std = x.varianceAlongRows().addScalar(1e-5).sqrt()
        x_hat = centred.divideBroadcastCols(std)
        y = x_hat.multiplyBroadcastRows(p["gamma"]).addRowVector(p["beta"])
        a = y.matmul(p["w1"]).addRowVector(p["b1"])
        f = a.geluActivation()
        o = f.matmul(p["w2"]).addRowVector(p["b2"]).add(x)
        logits = o.matmul(p["wh"]).addRowVector(p["bh"])
        losses.append(logits.crossEntropyLoss(targets))

        dl = logits.crossEntropyGradient(targets)
        grads = {"wh": o.transpose().matmul(dl), "bh": dl.sumRows()}
        do = dl.matmul(p["wh"].transpose())
        grads.update(w2=f.transpose().matmul(do), b2=do.sumRows())
        da = a.geluBackward(do.matmul(p["w2"].transpose()))
        grads.update(w1=y.transpose().matmul(da), b1=da.sumRows())
        dy = da.matmul(p["w1"].transpose())
        grads.update(gamma=dy.multiply(x_hat).sumRows(), beta=dy.sumRows())
        dx = Tensor.layerNormBackward(dy.multiplyBroadcastRows(p["gamma"]), x_hat, std, d).addInPlace(do)
        grads["emb"] = Tensor.zeros(s["vocab"], d)
        Tensor.scatterAddRows(grads["emb"], ids, dx)

        s["step"] += 1
        c1, c2 = 1.0 - 0.9 ** s["step"], 1.0 - 0.999 ** s["step"]
        for name, w in p.items():
            m, v = s["moments"][name]
            Tensor.adamWUpdate(w, grads[name], m, v, 3e-4, 0.9, 0.999, 1e-8, 0.01, c1, c2)
    return {"losses": np.array(losses, dtype=np.float32), "params": {n: t.numpy() for n, t in p.items()},
            "grads": {n: t.numpy() for n, t in grads.items()},
            "moments": {n: [m.numpy(), v.numpy()] for n, (m, v) in s["moments"].items()}}


def run(state):
    kind = state["kind"]
    if kind == "greedy":
        return TextGenerator.generate(state["model"], state["prompt_ids"], state["new"], 1.0, 1)
    if kind == "sampled":
        return TextGenerator.generate(state["model"], state["prompt_ids"], state["new"], state["temperature"], state["top_k"], state["seed"])
    if kind == "turns":
        return _turns(state)
    if kind == "steps":
        return _steps(state)
    if kind == "prompt":
        model = state["model"]
        model.reset()
        model.prefill(state["prompt_ids"], choose_next=False)
        return model.lastLogits()
    if kind == "score":
        return state["model"].forward(state["prompt_ids"])
    if kind == "attention":
        return _attention(state)
    if kind == "ffn":
        return _ffn(state)
    if kind == "train":
        return _train(state)
    dev = state["dev"]
    dev.write(state["xb"], state["x"])
    state["stream"].run()
    return dev.download(state["ob"], (state["rows"], state["d"]))


# ── what a pass cannot do without ────────────────────────────────────────────

_Q8 = 1.125        # bytes per Q8 weight with its share of the group's scale


def _block_weights(c):
    d, f = c["d"], c["dff"]
    if c["family"] == "gpt":
        return 4 * d * d + 2 * d * f
    if c["family"] in ("deepseek", "latent"):
        return 2 * d * c["q_rank"] + 3 * d * c["kv_rank"] + d * d + 3 * d * f
    return 4 * d * d + 3 * d * f


def _rows_work(c, n, before, heads_rows):
    """n rows behind `before` cached ones: block weights, cache and residual rows once; `heads_rows` rows of logits."""
    d, layers, head = c["d"], c["layers"], c["d"] * c["vocab"]
    per_position = 4 * (c["kv_rank"] if c["family"] == "latent" else 2 * d)
    bytes_ = _Q8 * (layers * _block_weights(c) + (head if heads_rows else 0)) + layers * per_position * (before + n) + 4 * n * d + 4 * heads_rows * c["vocab"]
    flops = 2 * n * layers * _block_weights(c) + 2 * heads_rows * head + layers * 4 * d * (n * before + n * (n + 1) / 2)
    if c["family"] == "latent":        # keys are rotated behind their up-projection, so each call expands them again
        flops += layers * 2 * before * c["kv_rank"] * d
    return np.array([bytes_, flops], dtype=np.float64)


def work(case):
    kind = case["kind"]
    if kind in ("greedy", "sampled", "turns", "steps", "prompt", "score"):
        n = case["prompt"]
        total = _rows_work(case, n, 0, n if kind == "score" else 1)
        at = n
        if kind in ("greedy", "sampled", "steps", "turns"):
            for _ in range(case["new"] if kind == "steps" else case["new"] - 1):
                total = total + _rows_work(case, 1, at, 1)
                at += 1
        for _ in range(case.get("turns", 0)):
            total = total + _rows_work(case, case["turn"] + 1, at, 1)
            at += case["turn"] + 1
            for _ in range(case["new"] - 1):
                total = total + _rows_work(case, 1, at, 1)
                at += 1
        return {"bytes": float(total[0]), "flops": float(total[1])}
    rows, d = case["rows"], case["d"]
    if kind == "attention":
        return {"bytes": 4.0 * (4 * d * d + 2 * rows * d), "flops": 8.0 * rows * d * d + 4.0 * rows * rows * d}
    if kind == "ffn":
        return {"bytes": 4.0 * (3 * d * case["dff"] + 2 * rows * d), "flops": 6.0 * rows * d * case["dff"]}
    if kind == "q8_ffn":
        return {"bytes": _Q8 * 3 * d * case["dff"] + 8.0 * rows * d, "flops": 6.0 * rows * d * case["dff"]}
    matrices = 2 * d * case["dff"] + d * case["vocab"]
    params = matrices + d * case["vocab"] + 4 * d + case["dff"] + case["vocab"]
    # per step: weights and both moments read and written (gradients can stay on the chip); at the end all four are read out
    return {"bytes": case["steps"] * 24.0 * params + 16.0 * params, "flops": case["steps"] * 6.0 * rows * matrices}


def tolerance(case):
    kind = case["kind"]
    if kind in ("greedy", "sampled", "turns"):
        return "exact"                              # token ids
    if kind in ("steps", "prompt", "score"):
        return {"rel": 1e-4, "max": 2e-3}           # 32-bit sums through all layers of a model
    if kind == "train":
        # 32-bit sums; AdamW's first steps take the sign of a gradient, so a value that sums to nearly nothing may step
        # the other way (2 x the learning rate a step, on values of 0.01 and more)
        return {"rel": 1e-4, "max": 0.3}
    return {"rel": 1e-5, "max": 1e-3}
