"""The timed work of this framework: what a program that runs a quantized model on one GPU asks of it.

Every case is one call (or one short run of calls) of `mongoose_amd.engine` -- the package's public mirror of the C ABI --
on a model of the benchmark configurations (`mongoose_amd.configs`) or a generic shape of the same family:

  generate  greedy decode of a prompt and a run of tokens                  HIPFusedInference.Generate
  sample    decode with the logits handed to the host, which chooses       HIPFusedInference.DecodeToken(.., logits)
  chat      a prompt in one batch, then a run of greedy tokens             HIPFusedInference.GeneratePrefill
  prefill   a prompt (or a further turn) in one batch, logits to the host  HIPFusedInference.Prefill
  stage     one stage of a pipeline over layers, hidden state in and out   HIPFusedInference.PartialStep
  stream    a token with the weights streamed from host memory             HIPStreamInfer.StreamForwardToken
  ops       a token composed by the caller from the per-op launches        K* functions
  gemm      several rows through one matrix                                KQ8Gemm / KQ8QuantizeActBatch + KQ4_0MatvecDP4ABatch
  load      fp32 weights quantized and uploaded, then the first token      SetWeight / quantize_q4_0 + SetWeightQ4_0

Weights, prompts and activations come from the seed.  A state holds a model of its own, as a program that serves several
models on one GPU does.  Matrix values are cut from a pool of normal samples at odd offsets (no two rows alike), row and
block scales vary from row to row as those of trained weights do.
"""
import math

import numpy as np
import torch

from mongoose_amd import configs
from mongoose_amd import engine as E

_STD = 0.02                       # standard deviation of the weights in the benchmark configurations


# ---------------------------------------------------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------------------------------------------------
def _model(s, layers=None, fmt=None, kvf16=False):
    return {"dim": s.dim, "heads": s.nHeads, "kvheads": s.nKVHeads, "hd": s.headDim, "ffn": s.ffnDim, "vocab": s.vocab,
            "layers": layers or s.nLayers, "eps": s.eps, "theta": s.theta, "bias": s.bias, "tied": s.tied,
            "fmt": fmt or s.fmt, "kvf16": kvf16}


def listed():
    C = configs
    return [
        # the smallest benchmark configuration: a four-layer model, 8 prompt tokens and 64 decoded ones; all launch latency
        dict(_model(C.TOY), name="toy-generate", op="generate", prompt=8, steps=64),
        # the headline: Q8 greedy decode of the 0.5B shape after a 16-token prompt
        dict(_model(C.QWEN), name="qwen-generate", op="generate", prompt=16, steps=64),
        # a client that samples on the host: the logits of every token cross to it, 1.1B shape, 600 positions in the cache
        dict(_model(C.TINYLLAMA), name="tinyllama-sample", op="sample", pos=600, steps=4),
        # the same at a long context, fp16 K/V rows, 8B shape (8 of its 32 layers: every layer is the same work)
        dict(_model(C.LLAMA3_8B, layers=8, kvf16=True), name="llama8b-sample-long", op="sample", pos=3900, steps=2),
        # a chat turn on 4-bit weights: an odd prompt of some hundred tokens in one batch, then a short answer
        dict(_model(C.QWEN_Q4), name="qwen-q4-chat", op="chat", prompt=301, steps=32),
        # a long prompt through the large shape, 8 of its 32 layers: the matrix cores' case
        dict(_model(C.LLAMA3_8B, layers=8), name="llama8b-prefill", op="prefill", pos=0, rows=512),
        # a short follow-up turn of a conversation: few rows behind a cache that already holds some
        dict(_model(C.QWEN), name="qwen-prefill-short", op="prefill", pos=200, rows=37),
        # the middle third of the 1.1B shape as one stage of a pipeline
        dict(_model(C.TINYLLAMA), name="tinyllama-stage", op="stage", first=7, last=15, pos=250),
        # 4-bit layers that stay in host memory, as for a model larger than the card's
        dict(_model(C.QWEN_Q4), name="qwen-q4-stream", op="stream", pos=33),
        # a caller with a decode loop of its own: four layers of the 1.1B shape from the per-op launches, 1,200 rows of cache
        dict(_model(C.TINYLLAMA, layers=4), name="tinyllama-ops", op="ops", pos=1199),
        # rows of a small batch against the 1.1B shape's gate matrix
        dict(name="gemm-77", op="gemm", fmt="q8", rows=77, n=5632, k=2048),
        # loading: four layers of the 0.5B shape and a 32,000-row head from fp32, then the first token
        dict(_model(C.QWEN._replace(vocab=32000), layers=4), name="qwen-load", op="load"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_model(rng, most_bytes):
    while True:
        if rng.random() < 0.4:
            s = rng.choice([configs.TOY, configs.QWEN, configs.TINYLLAMA, configs.QWEN_Q4, configs.LLAMA3_8B])
            m = _model(s, layers=rng.randint(1, min(s.nLayers, 24)), fmt=rng.choice(["q8", "q4_0"]), kvf16=rng.random() < 0.3)
        else:
            hd, kv, group = rng.choice([64, 64, 128]), rng.choice([1, 2, 3, 4, 5, 8]), rng.choice([1, 2, 3, 4, 6, 7, 8])
            dim = hd * kv * group
            if not 256 <= dim <= 4096:
                continue
            ffn = min(14336, 32 * max(8, _log(rng, 1.5 * dim, 5 * dim) // 32))
            m = {"dim": dim, "heads": kv * group, "kvheads": kv, "hd": hd, "ffn": ffn, "vocab": _log(rng, 250, 130000),
                 "layers": _log(rng, 1, 24), "eps": rng.choice([1e-5, 1e-6]), "theta": rng.choice([1e4, 5e5, 1e6]),
                 "bias": rng.random() < 0.5, "tied": rng.random() < 0.5, "fmt": rng.choice(["q8", "q8", "q4_0"]),
                 "kvf16": rng.random() < 0.3}
        if _layer_bytes(m) * m["layers"] + _head_bytes(m) <= most_bytes:
            return m


def draw(rng):
    op = rng.choice(["generate", "sample", "chat", "prefill", "prefill", "stage", "stream", "ops", "gemm", "load"])
    if op == "gemm":
        c = {"op": op, "fmt": rng.choice(["q8", "q8", "q4_0"]), "rows": _log(rng, 2, 600), "n": _log(rng, 200, 9000),
             "k": 32 * _log(rng, 8, 256)}
        if c["fmt"] == "q4_0":
            c["rows"] = min(c["rows"], 48)
        return c
    m = _draw_model(rng, {"load": 8e7, "stream": 2e8}.get(op, 1.2e9))
    token = _layer_bytes(m) * m["layers"] + _head_bytes(m)
    if op == "generate":
        m.update(prompt=_log(rng, 2, 40), steps=max(4, min(100, int(2e10 / token), _log(rng, 8, 100))))
    elif op == "sample":
        m.update(pos=_log(rng, 8, 4000), steps=rng.randint(1, 6))
    elif op == "chat":
        m.update(prompt=_log(rng, 16, 700), steps=max(4, min(40, int(1.5e10 / token))))
    elif op == "prefill":
        m.update(pos=rng.choice([0, 0, _log(rng, 8, 600)]), rows=_log(rng, 2, 1000))
    elif op == "stage":
        m["layers"] = max(2, m["layers"])
        first = rng.randint(0, m["layers"] - 2)
        m.update(first=first, last=rng.randint(first + 1, m["layers"] - 1), pos=_log(rng, 2, 1500))
    elif op == "stream":
        m.update(fmt="q4_0", pos=_log(rng, 2, 500))
    elif op == "ops":
        m["layers"] = min(m["layers"], 6)
        m.update(kvf16=False, pos=_log(rng, 8, 3000))
    elif op == "load":
        m["layers"] = min(m["layers"], 4)
    return dict(m, op=op)


# ---------------------------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------------------------------
def _mats(m):
    kv = m["kvheads"] * m["hd"]
    return {1: (m["dim"], m["dim"]), 2: (kv, m["dim"]), 3: (kv, m["dim"]), 7: (m["dim"], m["dim"]), 9: (m["ffn"], m["dim"]),
            10: (m["ffn"], m["dim"]), 11: (m["dim"], m["ffn"])}


def _mat_bytes(m, n, k):
    return n * k + 4 * n if m["fmt"] == "q8" else n * (k // 32) * 18


def _layer_bytes(m):
    return sum(_mat_bytes(m, n, k) for n, k in _mats(m).values()) + 8 * m["dim"]


def _layer_weights(m):
    return sum(n * k for n, k in _mats(m).values())


def _head_bytes(m):
    return _mat_bytes(m, m["vocab"], m["dim"]) + 4 * m["dim"]


def _kv_bytes(m, rows):          # K and V rows of one layer
    return rows * 2 * m["kvheads"] * m["hd"] * (2 if m["kvf16"] else 4)


def _attn_flops(m, pos):         # scores and P.V of one query at position pos, one layer
    return 4.0 * (pos + 1) * m["dim"]


def work(case):
    m, op = case, case["op"]
    if op == "gemm":
        t, n, k = m["rows"], m["n"], m["k"]
        return {"bytes": 4.0 * t * (k + n) + _mat_bytes(m, n, k), "flops": 2.0 * t * n * k}
    L, lb, hb, lw, hw = m["layers"], _layer_bytes(m), _head_bytes(m), _layer_weights(m), m["vocab"] * m["dim"]
    if op == "load":             # fp32 in, quantized out to the card, then a token
        w = L * lw + hw
        return {"bytes": 4.0 * w + 2.0 * (L * lb + hb), "flops": 2.0 * w}
    steps = range(0)
    rows = 0                     # prompt rows that go through the layers together
    p0 = m.get("pos", 0)
    if op == "generate":
        rows, p0, steps = m["prompt"] - 1, 0, range(m["prompt"] - 1, m["prompt"] - 1 + m["steps"])
    elif op == "chat":
        rows, p0, steps = m["prompt"], 0, range(m["prompt"], m["prompt"] + m["steps"] - 1)
    elif op == "sample":
        steps = range(p0, p0 + m["steps"])
    elif op == "prefill":
        rows = m["rows"]
    elif op in ("stream", "ops"):
        steps = range(p0, p0 + 1)
    elif op == "stage":
        n = m["last"] - m["first"]
        return {"bytes": n * (lb + _kv_bytes(m, p0 + 1)) + 8.0 * m["dim"], "flops": n * (2.0 * lw + _attn_flops(m, p0))}
    b = sum(L * (lb + _kv_bytes(m, p + 1)) + hb for p in steps)
    f = sum(L * (2.0 * lw + _attn_flops(m, p)) + 2.0 * hw for p in steps)
    if rows:
        b += L * (lb + _kv_bytes(m, p0 + rows))
        f += L * (2.0 * lw * rows + sum(_attn_flops(m, p0 + r) for r in range(rows)))
        if op in ("chat", "prefill"):
            b, f = b + hb, f + 2.0 * hw
    if op in ("sample", "prefill", "stream", "ops"):
        b += 4.0 * m["vocab"] * max(1, len(steps))
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    op = case["op"]
    if op in ("generate", "chat"):
        return {"differ": 0.01}                       # token ids
    if op == "gemm":                                  # q8: activations as two bf16 terms (2^-16); q4_0: whole-number sums, fp32 across blocks
        return {"rel": 3e-5, "max": 3e-4}
    if case["kvf16"]:
        return {"rel": 1e-3, "max": 1e-2}             # a K/V row's last bit decides how it rounds to fp16
    if op == "prefill" or (op == "sample" and case["pos"] > 0):
        return {"rel": 2e-4, "max": 2e-3}             # the rows in the cache come from two-term bf16 products, layer after layer
    return {"rel": 5e-5, "max": 5e-4}                 # fp32 sums, layer after layer


# ---------------------------------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------------------------------
_POOL = 4_194_301                                     # samples in a pool (odd, so that rows cut from it fall differently)


class _Weights:
    """Matrices, scales and vectors of one seed."""

    def __init__(self, seed):
        self.rng = np.random.default_rng([seed, 4711])
        self.normal = self.rng.standard_normal(_POOL, dtype=np.float32)
        self.at = 0

    def cut(self, pool, n):
        """n items of the pool, starting somewhere else each time."""
        self.at = (self.at + 1_299_709) % len(pool)
        if self.at + n <= len(pool):
            return pool[self.at:self.at + n]
        return np.resize(np.concatenate([pool[self.at:], pool[:self.at]]), n)

    def vec(self, n, mean=0.0):
        return (mean + _STD * self.cut(self.normal, n)).astype(np.float32)

    def f32(self, rows, cols):
        a = self.cut(self.normal, rows * cols).reshape(rows, cols)
        return a * (_STD * self.spread(rows))[:, None]

    def spread(self, rows, by=0.25):
        return np.exp(by * self.rng.standard_normal(rows, dtype=np.float32))

    def q8(self, rows, cols, by=0.25):
        if not hasattr(self, "int8"):
            self.int8 = np.clip(np.rint(self.normal * 36.0), -127, 127).astype(np.int8)
        return self.cut(self.int8, rows * cols).reshape(rows, cols), (_STD / 36.0 * self.spread(rows, by)).astype(np.float32)

    def q4(self, rows, cols, by=0.25):
        """GGUF block_q4_0: fp16 d, 16 bytes of nibbles."""
        if not hasattr(self, "blocks"):
            n = _POOL // 32
            b = np.empty((n, 18), np.uint8)
            d = (_STD / 2.7 * self.spread(n, by)) * np.where(self.rng.random(n) < 0.5, -1, 1)
            b[:, :2] = d.astype(np.float16).view(np.uint8).reshape(n, 2)
            nib = np.clip(np.rint(self.normal[:n * 32] * 2.7 + 8), 0, 15).astype(np.uint8).reshape(n, 2, 16)
            b[:, 2:] = nib[:, 0] | (nib[:, 1] << 4)
            self.blocks = b
        n = rows * (cols // 32)
        self.at = (self.at + 1_299_709) % len(self.blocks)
        if self.at + n <= len(self.blocks):
            return self.blocks[self.at:self.at + n].reshape(-1)
        return np.resize(np.concatenate([self.blocks[self.at:], self.blocks[:self.at]]).reshape(-1), n * 18)


def _context(m, W, maxSeq, first=0, last=None, set_matrices=True, streamed=False):
    """A context with its weights: layers first .. last - 1 and, behind the last layer, the head."""
    eng = E.NewHIP(0)
    last = m["layers"] if last is None else last
    f = E.NewHIPFusedInference(eng, m["dim"], m["kvheads"] * m["hd"], m["hd"], m["heads"], m["kvheads"], m["ffn"], m["vocab"],
                               m["layers"], maxSeq, m["theta"], m["eps"])
    assert f is not None, E.last_error()
    if m["kvf16"]:
        f.SetKVFormat(1)
    f.SetLayerRange(first, last)

    def matrix(idx, rows, cols, by=0.25):
        if m["fmt"] == "q8":
            q, sc = W.q8(rows, cols, by)
            rc = f.SetWeightQ8(idx, q, sc)
        else:
            rc = f.SetWeightQ4_0(idx, W.q4(rows, cols, by))
        assert rc == 0, E.last_error()

    kv = m["kvheads"] * m["hd"]
    for l in range(first, last):
        if streamed:
            break
        f.SetWeight(l * 12, W.vec(m["dim"], 1.0))
        f.SetWeight(l * 12 + 8, W.vec(m["dim"], 1.0))
        if m["bias"]:
            for k, n in ((4, m["dim"]), (5, kv), (6, kv)):
                f.SetWeight(l * 12 + k, W.vec(n))
        if set_matrices:
            for k, (rows, cols) in _mats(m).items():
                matrix(l * 12 + k, rows, cols)
    if last == m["layers"]:
        f.SetWeight(m["layers"] * 12, W.vec(m["dim"], 1.0))
        if set_matrices:
            matrix(m["layers"] * 12 + 1, m["vocab"], m["dim"], 0.4)
        if not m["tied"]:
            half = (W.normal * np.float32(_STD)).astype(np.float16)
            f.SetEmbeddingF16(W.cut(half, m["vocab"] * m["dim"]))
    return f


def prepare(case, seed):
    m, op = case, case["op"]
    if op == "gemm":
        return _prepare_gemm(m, seed)
    if op == "ops":
        return _prepare_ops(m, seed)
    W = _Weights(seed)
    st = {"op": op, "m": m}
    tokens = lambda n: W.rng.integers(0, m["vocab"], n).astype(np.int32)  # noqa: E731
    if op in ("generate", "chat"):
        st["prompt"] = tokens(m["prompt"])
        st["f"] = _context(m, W, m["prompt"] + m["steps"])
    elif op == "sample":
        f = st["f"] = _context(m, W, m["pos"] + m["steps"] + 64)
        st["tokens"] = tokens(m["steps"])
        st["logits"] = np.zeros((m["steps"], m["vocab"]), np.float32)
        rc = f.Prefill(tokens(m["pos"]), 0)[0]
        assert rc == 0, E.last_error()
    elif op == "prefill":
        f = st["f"] = _context(m, W, m["pos"] + m["rows"] + 64)
        st["tokens"] = tokens(m["rows"])
        if m["pos"]:
            rc = f.Prefill(tokens(m["pos"]), 0)[0]
            assert rc == 0, E.last_error()
    elif op == "stage":
        f = st["f"] = _context(m, W, m["pos"] + 64, first=m["first"], last=m["last"])
        st["hidden"] = W.cut(W.normal, m["dim"]).copy()
        st["out"] = np.zeros(m["dim"], np.float32)
        for pos in range(max(0, m["pos"] - 64), m["pos"]):      # (rows before these stay zero, as in a fresh cache)
            f.PartialStep(W.cut(W.normal, m["dim"]), pos, m["first"], m["last"], None, None)
    elif op == "stream":
        f = st["f"] = _context(m, W, m["pos"] + 64, streamed=True)
        st["s"] = f.StreamBuild()
        assert st["s"] is not None, E.last_error()
        ptrs, sizes, kv = [], [], m["kvheads"] * m["hd"]
        for _ in range(m["layers"]):
            mats = {k: W.q4(r, c).copy() for k, (r, c) in _mats(m).items()}
            vecs = {0: W.vec(m["dim"], 1.0), 8: W.vec(m["dim"], 1.0)}
            if m["bias"]:
                vecs.update({4: W.vec(m["dim"]), 5: W.vec(kv), 6: W.vec(kv)})
            ptrs += [mats.get(k, vecs.get(k)) for k in range(12)]
            sizes += [mats[k].size for k in (1, 2, 3, 7, 9, 10, 11)]
        st["ptrs"], st["sizes"] = ptrs, sizes
        st["hidden"] = (_STD * W.cut(W.normal, m["dim"])).astype(np.float32)
        st["logits"] = np.zeros(m["vocab"], np.float32)
        for pos in range(max(0, m["pos"] - 4), m["pos"]):       # (rows before these stay zero, as in a fresh cache)
            st["s"].StreamForwardToken(pos, _STD * W.cut(W.normal, m["dim"]), m["layers"], ptrs, sizes, None)
    elif op == "load":
        st["f"] = _context(m, W, 64, set_matrices=False)
        st["mats"] = {l * 12 + k: W.f32(r, c) for l in range(m["layers"]) for k, (r, c) in _mats(m).items()}
        st["mats"][m["layers"] * 12 + 1] = W.f32(m["vocab"], m["dim"])
        st["token"] = int(tokens(1)[0])
        st["logits"] = np.zeros(m["vocab"], np.float32)
    return st


def _prepare_gemm(m, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    t, n, k = m["rows"], m["n"], m["k"]
    st = {"op": "gemm", "m": m, "out": torch.empty(t, n, device="cuda"), "act": torch.randn(t, k, device="cuda", generator=g)}
    E.NewHIP(0)
    if m["fmt"] == "q8":
        st["w"] = torch.randint(-127, 128, (n, k), device="cuda", generator=g, dtype=torch.int8)
        st["scales"] = _STD / 73 * torch.exp(0.25 * torch.randn(n, device="cuda", generator=g))
        st["bias"] = _STD * torch.randn(n, device="cuda", generator=g)
        st["ws"] = torch.empty(4 * ((t + 127) // 128 * 128) * ((k + 63) // 64 * 64), dtype=torch.uint8, device="cuda")
    else:
        st["w"] = torch.from_numpy(_Weights(seed).q4(n, k).copy()).cuda()
        st["q"] = torch.empty(t * (k // 32) * 40, dtype=torch.uint8, device="cuda")
    return st


def _prepare_ops(m, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    E.NewHIP(0)
    kv, rows = m["kvheads"] * m["hd"], m["pos"] + 1
    W = _Weights(seed) if m["fmt"] != "q8" else None
    rnd = lambda *shape: torch.randn(*shape, device="cuda", generator=g)  # noqa: E731

    def matrix(n, k):
        if m["fmt"] == "q8":
            return (torch.randint(-127, 128, (n, k), device="cuda", generator=g, dtype=torch.int8),
                    _STD / 73 * torch.exp(0.25 * rnd(n)), n, k)
        return (torch.from_numpy(W.q4(n, k).copy()).cuda(), None, n, k)

    layers = []
    for _ in range(m["layers"]):
        L = {k: matrix(*nk) for k, nk in _mats(m).items()}
        L.update(norm1=1 + _STD * rnd(m["dim"]), norm2=1 + _STD * rnd(m["dim"]), K=rnd(rows, kv), V=rnd(rows, kv))
        if m["bias"]:
            L.update(bq=_STD * rnd(m["dim"]), bk=_STD * rnd(kv), bv=_STD * rnd(kv))
        layers.append(L)
    j = torch.arange(m["hd"] // 2, device="cuda", dtype=torch.float64)
    angle = m["pos"] * m["theta"] ** (-2 * j / m["hd"])
    new = lambda n: torch.empty(n, device="cuda")  # noqa: E731
    return {"op": "ops", "m": m, "layers": layers, "norm": 1 + _STD * rnd(m["dim"]), "head": matrix(m["vocab"], m["dim"]),
            "embed": _STD * rnd(64, m["dim"]), "token": torch.randint(0, 64, (1,), device="cuda", generator=g, dtype=torch.int32),
            "cos": torch.cos(angle).float(), "sin": torch.sin(angle).float(), "x": new(m["dim"]), "h": new(m["dim"]),
            "q": new(m["dim"]), "k": new(kv), "v": new(kv), "a": new(m["dim"]), "p": new(m["dim"]), "gate": new(m["ffn"]),
            "up": new(m["ffn"]), "mid": new(m["ffn"]), "logits": new(m["vocab"])}


# ---------------------------------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------------------------------
def run(st):
    return _RUN[st["op"]](st, st["m"])


def _generate(st, m):
    rc, toks = st["f"].Generate(st["prompt"], m["steps"], useGraph=True)
    assert rc == 0, E.last_error()
    return toks


def _chat(st, m):
    rc, toks = st["f"].GeneratePrefill(st["prompt"], m["steps"])
    assert rc == 0, E.last_error()
    return toks


def _sample(st, m):
    f, logits = st["f"], st["logits"]
    for i in range(m["steps"]):
        rc, _ = f.DecodeToken(int(st["tokens"][i]), m["pos"] + i, logits[i])
        assert rc == 0, E.last_error()
    return logits


def _prefill(st, m):
    rc, nxt, logits, _ = st["f"].Prefill(st["tokens"], m["pos"], wantLogits=True)
    assert rc == 0, E.last_error()
    return logits


def _stage(st, m):
    rc = st["f"].PartialStep(st["hidden"], m["pos"], m["first"], m["last"], st["out"], None)
    assert rc == 0, E.last_error()
    return st["out"]


def _stream(st, m):
    rc = st["s"].StreamForwardToken(m["pos"], st["hidden"], m["layers"], st["ptrs"], st["sizes"], st["logits"])
    assert rc == 0, E.last_error()
    return st["logits"]


def _load(st, m):
    f = st["f"]
    for idx, w in st["mats"].items():
        rc = f.SetWeight(idx, w) if m["fmt"] == "q8" else f.SetWeightQ4_0(idx, E.quantize_q4_0(w))
        assert rc == 0, E.last_error()
    rc, _ = f.DecodeToken(st["token"], 0, st["logits"])
    assert rc == 0, E.last_error()
    return st["logits"]


def _gemm(st, m):
    act, w, out = st["act"].data_ptr(), st["w"].data_ptr(), st["out"]
    t, n, k = m["rows"], m["n"], m["k"]
    if m["fmt"] == "q8":
        E.KQ8Gemm(act, w, st["scales"].data_ptr(), st["bias"].data_ptr(), out.data_ptr(), t, n, k, 0, st["ws"].data_ptr(),
                  st["ws"].numel())
    else:
        q = st["q"].data_ptr()
        E.KQ8QuantizeActBatch(act, q, k, t)
        E.KQ4_0MatvecDP4ABatch(w, q, out.data_ptr(), n, k, t)
    return out


def _ops(st, m):
    p = {k: v.data_ptr() for k, v in st.items() if isinstance(v, torch.Tensor)}
    dim, ffn, hd, kv, pos = m["dim"], m["ffn"], m["hd"], m["kvheads"] * m["hd"], m["pos"]

    def mul(mat, act, out):
        w, sc, n, k = mat
        if sc is not None:
            E.KQ8MatvecRowScale(act, w.data_ptr(), sc.data_ptr(), out, n, k)
        else:
            E.KQ4_0Matvec(act, w.data_ptr(), out, n, k)

    E.KEmbedGather2(p["x"], p["embed"], p["token"], 1, dim)
    for L in st["layers"]:
        K, V = L["K"].data_ptr(), L["V"].data_ptr()
        E.KRMSNormOutEps(p["x"], p["h"], L["norm1"].data_ptr(), 1, dim, m["eps"])
        mul(L[1], p["h"], p["q"])
        mul(L[2], p["h"], p["k"])
        mul(L[3], p["h"], p["v"])
        if m["bias"]:
            E.KAddInPlace(p["q"], L["bq"].data_ptr(), dim)
            E.KAddInPlace(p["k"], L["bk"].data_ptr(), kv)
            E.KAddInPlace(p["v"], L["bv"].data_ptr(), kv)
        E.KRoPE(p["q"], p["cos"], p["sin"], 1, dim, hd, m["heads"])
        E.KRoPE(p["k"], p["cos"], p["sin"], 1, kv, hd, m["kvheads"])
        E.KKVCacheWrite(K, p["k"], pos, kv)
        E.KKVCacheWrite(V, p["v"], pos, kv)
        E.KDecodeAttention(p["q"], K, V, p["a"], pos + 1, dim, kv, m["heads"], m["kvheads"])
        mul(L[7], p["a"], p["p"])
        E.KAddInPlace(p["x"], p["p"], dim)
        E.KRMSNormOutEps(p["x"], p["h"], L["norm2"].data_ptr(), 1, dim, m["eps"])
        mul(L[9], p["h"], p["gate"])
        mul(L[10], p["h"], p["up"])
        E.KSiLUGateMul(p["gate"], p["up"], p["mid"], ffn)
        mul(L[11], p["mid"], p["p"])
        E.KAddInPlace(p["x"], p["p"], dim)
    E.KRMSNormOutEps(p["x"], p["h"], p["norm"], 1, dim, m["eps"])
    mul(st["head"], p["h"], p["logits"])
    return [st["x"], st["logits"]]


_RUN = {"generate": _generate, "sample": _sample, "chat": _chat, "prefill": _prefill, "stage": _stage, "stream": _stream,
        "ops": _ops, "gemm": _gemm, "load": _load}
