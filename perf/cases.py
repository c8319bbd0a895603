"""The framework's performance cases: what a program that serves or scores text with it has it do.

A case is a dict of plain values. Its `kind` says which public entry points a pass calls:

* decode    one token through a loaded model (`Model.forward`): the loop of an interactive program;
* prompt    a prompt into the KV cache (`Model.prefill`), its last token by `Model.forward`, whose
            logits start the answer;
* score     every position's logits of a text (`Model.prefill(want_logits=True)`): perplexity, ranking;
* batch     one step of n sequences at their own positions (`Batch.forward`): a server's step;
* generate  n sampled tokens on the device (`Model.sample`, the command line's default temperature and
            nucleus), then the next logits;
* matmul    `qmh_matmul_nt` on device matrices (f32, the reference bench's GEMM row);
* matvec    `qmh_matvec`, or `qmh_rmsnorm_matvec` where a gain is given, on an uploaded weight;
* quantize  `qmh_quantize_rows_q8` / `_q4` of a device matrix (a converter's work).

Model shapes are those of the framework's workloads c1 to c5 (`quillm_amd.WORKLOADS`); c4 and c5 run
with fewer layers (a layer repeats, and four 7B-shaped ones already exceed every cache). Weights are
random, N(0, 0.02), quantized on the GPU when a state is prepared; all inputs come from the seed.

The framework's contract is bitwise: a result is the float that the scalar reference's order of
operations gives, whatever the kernel. So every tolerance is "exact".
"""
import ctypes
import math

import numpy as np
import torch

import quillm_amd as q

# dim, hidden_dim, layers, heads, kv heads, vocabulary (c1 to c5 of quillm_amd.WORKLOADS; c4 and c5 cut in depth)
SHAPES = {
    "c1": (288, 768, 6, 6, 6, 32000),
    "c2": (288, 768, 6, 6, 2, 32000),
    "c3": (768, 2048, 12, 12, 12, 32000),
    "c4": (2048, 5632, 8, 32, 4, 32000),
    "c5": (4096, 11008, 4, 32, 32, 32000),
}
THETA, EPS = 10000.0, 1e-5


def listed():
    return [
        # the smallest call: one token of a 15M-parameter model, all latency and launches
        {"name": "decode small", "kind": "decode", "shape": "c1", "wtype": "q8_0", "pos": 37},
        # the headline: a 7B-shaped Q4_0 model answering, mid-conversation
        {"name": "decode 7b", "kind": "decode", "shape": "c5", "wtype": "q4_0", "pos": 575},
        # a long conversation on a grouped-query model, past the one-launch attention's limit
        {"name": "decode gqa long", "kind": "decode", "shape": "c4", "wtype": "q4_0", "pos": 1531},
        # the headline prompt: 512 tokens through the 7B-shaped Q4_0 layers
        {"name": "prompt 7b", "kind": "prompt", "shape": "c5", "wtype": "q4_0", "n": 513},
        # a long document into a grouped-query model: several passes, attention over a growing context
        {"name": "prompt gqa long", "kind": "prompt", "shape": "c4", "wtype": "q4_0", "n": 1901},
        # a short text scored with the 7B-shaped Q8_0 model: every position's logits, an odd token count
        {"name": "score short", "kind": "score", "shape": "c5", "wtype": "q8_0", "n": 33},
        # a server's step: 16 conversations on the 7B-shaped Q4_0 model, each at its own position
        {"name": "batch 7b", "kind": "batch", "shape": "c5", "wtype": "q4_0", "n": 16, "most": 448},
        # a busy server's step: 96 short conversations on the grouped-query model
        {"name": "batch gqa wide", "kind": "batch", "shape": "c4", "wtype": "q8_0", "n": 96, "most": 160},
        # text generation with the command line's defaults (temperature 0.8, top-p 0.95)
        {"name": "generate", "kind": "generate", "shape": "c3", "wtype": "q8_0", "n": 16, "pos": 128},
        # the reference bench's f32 matmul, at a size with remainders on every side
        {"name": "matmul", "kind": "matmul", "m": 1000, "n": 1090, "k": 1500},
        # an unquantized layer's matvec (7B attention width)
        {"name": "matvec f32", "kind": "matvec", "wtype": "f32", "rows": 4096, "cols": 4096, "norm": False},
        # a converter turning a 7B attention matrix into Q4_0 rows
        {"name": "quantize", "kind": "quantize", "wtype": "q4_0", "rows": 4096, "cols": 4096},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prompt", "prompt", "score", "batch", "batch", "generate", "matmul", "matvec",
                       "quantize"])
    shape, wtype = rng.choice(sorted(SHAPES)), rng.choice(["q4_0", "q8_0"])
    if kind == "decode":
        return {"kind": kind, "shape": shape, "wtype": wtype, "pos": _log(rng, 1, 1900)}
    if kind == "prompt":
        most = {"c5": 512, "c4": 1900}.get(shape, 1900)
        return {"kind": kind, "shape": shape, "wtype": wtype, "n": _log(rng, 2, most)}
    if kind == "score":
        return {"kind": kind, "shape": shape, "wtype": wtype, "n": _log(rng, 1, 96)}
    if kind == "batch":
        n = _log(rng, 1, 96)
        return {"kind": kind, "shape": shape, "wtype": wtype, "n": n, "most": _log(rng, 8, 448 if n <= 16 else 160)}
    if kind == "generate":
        return {"kind": kind, "shape": shape, "wtype": wtype, "n": rng.randint(1, 16), "pos": _log(rng, 1, 600)}
    if kind == "matmul":
        return {"kind": kind, "m": _log(rng, 16, 1100), "n": _log(rng, 16, 1100), "k": _log(rng, 16, 1500)}
    if kind == "matvec":
        wtype = rng.choice(["f32", "q8_0", "q4_0"])
        return {"kind": kind, "wtype": wtype, "rows": _log(rng, 64, 4096), "cols": _log(rng, 64, 4096),
                "norm": rng.choice([False, True])}
    return {"kind": kind, "wtype": wtype, "rows": _log(rng, 64, 4096), "cols": _log(rng, 64, 4096)}


# ------------------------------------------------------------------------------------- weights and models

def _gen(seed, *what):
    g = torch.Generator(device="cuda")
    g.manual_seed((hash((int(seed),) + what) & ((1 << 62) - 1)))
    return g


def _blocks(w, wtype):
    """Rows of the .qlm / qm_tensor layout: per 32 values an fp16 scale, then int8 codes (Q8_0) or nibbles (Q4_0)."""
    rows, cols = w.shape
    if wtype == "f32":
        return w.contiguous().view(torch.uint8).reshape(rows, -1)
    nb = (cols + 31) // 32
    b = torch.zeros(rows, nb * 32, device=w.device)
    b[:, :cols] = w
    b = b.view(rows, nb, 32)
    top = 127.0 if wtype == "q8_0" else 7.0
    d = (b.abs().amax(2, keepdim=True) / top).half()
    dd = d.float()
    c = torch.where(dd > 0, torch.round(b / torch.where(dd > 0, dd, torch.ones_like(dd))), torch.zeros_like(b))
    if wtype == "q8_0":
        code = c.clamp(-127, 127).to(torch.int8).view(torch.uint8)
    else:
        u = (c.clamp(-8, 7) + 8).to(torch.uint8)
        code = u[:, :, 0::2] | (u[:, :, 1::2] << 4)
    return torch.cat([d.view(torch.uint8), code], 2).reshape(rows, -1)


def _values(raw, cols, wtype):
    """The float64 values of _blocks' rows."""
    rows = raw.shape[0]
    if wtype == "f32":
        return raw.contiguous().view(torch.float32).reshape(rows, cols).double()
    bs = 34 if wtype == "q8_0" else 18
    b = raw.view(rows, -1, bs)
    d = b[:, :, :2].contiguous().view(torch.float16).double()
    if wtype == "q8_0":
        c = b[:, :, 2:].contiguous().view(torch.int8).double()
    else:
        n = b[:, :, 2:]
        c = torch.stack([n & 15, n >> 4], 3).reshape(rows, b.shape[1], 32).double() - 8
    return (c * d).reshape(rows, -1)[:, :cols]


def _shapes(shape):
    dim, hidden, _, heads, kv, _ = SHAPES[shape]
    kvd = dim // heads * kv
    return [("wq", dim, dim), ("wk", kvd, dim), ("wv", kvd, dim), ("wo", dim, dim), ("w1", hidden, dim),
            ("w2", dim, hidden), ("w3", hidden, dim)]


def _weights(case, seed):
    """{name: raw rows or float vector, on the GPU}, layer by layer."""
    dim, _, layers, _, _, vocab = SHAPES[case["shape"]]
    kind = sorted(SHAPES).index(case["shape"])
    g = _gen(seed, 1, kind)

    def mat(rows, cols):
        return _blocks(torch.randn(rows, cols, device="cuda", generator=g) * 0.02, case["wtype"])

    def gain():
        return 1.0 + 0.1 * torch.randn(dim, device="cuda", generator=g)

    top = {"tok_embd": mat(vocab, dim), "norm": gain(), "output": mat(vocab, dim)}
    lay = []
    for _ in range(layers):
        one = {name: mat(rows, cols) for name, rows, cols in _shapes(case["shape"])}
        one["attn_norm"], one["ffn_norm"] = gain(), gain()
        lay.append(one)
    return top, lay


def _model(case, seed, max_seq):
    """The model on the device, from host tensors as a loader that holds a file hands them over (qmh_model_create)."""
    dim, hidden, layers, heads, kv, vocab = SHAPES[case["shape"]]
    top, lay = _weights(case, seed)
    keep = []

    def view(t, rows, cols):
        h = t.cpu()
        keep.append(h)
        v = q.TensorView()
        v.data = h.data_ptr()
        if cols:
            v.dtype, v.ndim = q.DTYPES[case["wtype"]], 2
            v.ne[0], v.ne[1] = rows, cols
        else:
            v.dtype, v.ndim = q.F32, 1
            v.ne[0] = rows
        return v

    sizes = {name: (rows, cols) for name, rows, cols in _shapes(case["shape"])}
    order = ["attn_norm", "wq", "wk", "wv", "wo", "ffn_norm", "w1", "w2", "w3"]
    views = (q.TensorView * (9 * layers))()
    for i, one in enumerate(lay):
        for k, name in enumerate(order):
            views[9 * i + k] = view(one[name], *sizes.get(name, (dim, 0)))
    e, n, o = view(top["tok_embd"], vocab, dim), view(top["norm"], dim, 0), view(top["output"], vocab, dim)
    del top, lay
    cfg = q.QmhConfig(dim, hidden, layers, heads, kv, vocab, max_seq, THETA, EPS)
    h = q.load_library().qmh_model_create(ctypes.byref(cfg), ctypes.byref(e), ctypes.byref(n), ctypes.byref(o), views)
    if not h:
        raise q.QmhError("qmh_model_create: " + q.last_error())
    return q.Model(h)


def _tokens(case, seed, *size):
    rng = np.random.default_rng([int(seed), 7])
    return rng.integers(2, SHAPES[case["shape"]][5], size).astype(np.int32)


def _batch_state(case, seed):
    """The sequences' tokens [n, most + 1] and the position of each one's step."""
    toks = _tokens(case, seed, case["n"], case["most"] + 1)
    rng = np.random.default_rng([int(seed), 8])
    pos = rng.integers(case["most"] // 2, case["most"] + 1, case["n"]).astype(np.int32)
    return toks, pos


def _max_seq(case):
    most = {"decode": lambda: case["pos"] + 1, "prompt": lambda: case["n"], "score": lambda: case["n"],
            "batch": lambda: case["most"] + 1, "generate": lambda: case["pos"] + 512}[case["kind"]]()
    return max(256, (most + 127) // 128 * 128)


# ------------------------------------------------------------------------------------- the interface

def prepare(case, seed):
    q.init(0)
    kind = case["kind"]
    if kind in ("matmul", "matvec", "quantize"):
        return _prepare_op(case, seed)
    m = _model(case, seed, _max_seq(case))
    s = {"kind": kind, "model": m}
    if kind == "decode":
        t = _tokens(case, seed, case["pos"] + 1)
        m.prefill(t[:-1], 0)
        s["token"], s["pos"] = int(t[-1]), case["pos"]
    elif kind in ("prompt", "score"):
        s["tokens"] = _tokens(case, seed, case["n"])
    elif kind == "batch":
        toks, pos = _batch_state(case, seed)
        b = q.Batch(m, case["n"])
        for p in range(int(pos.max())):  # the conversations so far
            b.forward(toks[:, p], np.full(case["n"], p, np.int32), want_logits=False)
        s["batch"], s["pos"] = b, pos
        s["tokens"] = np.ascontiguousarray(toks[np.arange(case["n"]), pos])
    else:
        t = _tokens(case, seed, case["pos"] + 1)
        m.prefill(t[:-1], 0)
        s["sampler"] = q.Sampler(SHAPES[case["shape"]][5], 0.8, 0, 0.95, int(seed) + 1)
        s["token"], s["pos"], s["n"] = int(t[-1]), case["pos"], case["n"]
    return s


def _prepare_op(case, seed):
    g = _gen(seed, 2)
    s = {"kind": case["kind"]}
    if case["kind"] == "matmul":
        s["a"] = torch.randn(case["m"], case["k"], device="cuda", generator=g)
        s["b"] = torch.randn(case["n"], case["k"], device="cuda", generator=g)
        s["c"] = torch.empty(case["m"], case["n"], device="cuda")
    elif case["kind"] == "matvec":
        raw, x, gain = _matvec_inputs(case, g)
        host = raw.cpu()
        w = q.load_library().qmh_weight_upload(q.DTYPES[case["wtype"]], case["rows"], case["cols"], host.data_ptr())
        if not w:
            raise q.QmhError("qmh_weight_upload: " + q.last_error())
        s["w"], s["x"], s["gain"] = _Weight(w), x, gain
        s["y"] = torch.empty(case["rows"], device="cuda")
    else:
        s["x"] = torch.randn(case["rows"], case["cols"], device="cuda", generator=g) * 0.02
        bs = 34 if case["wtype"] == "q8_0" else 18
        s["y"] = torch.empty(case["rows"], (case["cols"] + 31) // 32 * bs, device="cuda", dtype=torch.uint8)
        s["fn"] = "qmh_quantize_rows_q8" if case["wtype"] == "q8_0" else "qmh_quantize_rows_q4"
    torch.cuda.synchronize()  # the library has a stream of its own
    return s


class _Weight:
    """An uploaded weight, freed with the state that holds it."""

    def __init__(self, handle):
        self.handle = handle

    def __del__(self):
        q.sync()
        q.load_library().qmh_weight_free(self.handle)


def _matvec_inputs(case, g):
    raw = _blocks(torch.randn(case["rows"], case["cols"], device="cuda", generator=g) * 0.02, case["wtype"])
    x = torch.randn(case["cols"], device="cuda", generator=g)
    gain = 1.0 + 0.1 * torch.randn(case["cols"], device="cuda", generator=g) if case["norm"] else None
    return raw, x, gain


def _ok(rc):
    if rc:
        raise q.QmhError(q.last_error())


def run(s):
    kind = s["kind"]
    # forward's logits are a view of the model's own memory, valid until its next call: a program
    # that keeps them copies them
    if kind == "decode":
        return s["model"].forward(s["token"], s["pos"]).copy()
    if kind == "prompt":
        t = s["tokens"]
        s["model"].prefill(t[:-1], 0)
        return s["model"].forward(int(t[-1]), len(t) - 1).copy()
    if kind == "score":
        return s["model"].prefill(s["tokens"], 0, want_logits=True)
    if kind == "batch":
        return s["batch"].forward(s["tokens"], s["pos"])
    if kind == "generate":
        ids = s["model"].sample(s["sampler"], s["token"], s["pos"], s["n"])
        return {"ids": ids, "logits": s["model"].forward(int(ids[-1]), s["pos"] + s["n"]).copy()}
    lib = q.load_library()
    if kind == "matmul":
        a, b, c = s["a"], s["b"], s["c"]
        _ok(lib.qmh_matmul_nt(a.data_ptr(), b.data_ptr(), c.data_ptr(), a.shape[0], b.shape[0], a.shape[1], None))
        return c
    if kind == "matvec":
        if s["gain"] is not None:
            _ok(lib.qmh_rmsnorm_matvec(s["w"].handle, s["x"].data_ptr(), s["gain"].data_ptr(), EPS, s["y"].data_ptr(),
                                       None, None))
        else:
            _ok(lib.qmh_matvec(s["w"].handle, s["x"].data_ptr(), s["y"].data_ptr(), None, None))
        return s["y"]
    _ok(getattr(lib, s["fn"])(s["x"].data_ptr(), s["y"].data_ptr(), s["x"].shape[0], s["x"].shape[1], None))
    return s["y"]


def _row_bytes(cols, wtype):
    return 4 * cols if wtype == "f32" else (cols + 31) // 32 * (34 if wtype == "q8_0" else 18)


def work(case):
    kind = case["kind"]
    if kind == "matmul":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 4 * (m * k + n * k + m * n), "flops": 2 * m * n * k}
    if kind == "matvec":
        r, c = case["rows"], case["cols"]
        return {"bytes": r * _row_bytes(c, case["wtype"]) + 4 * (r + c * (2 if case["norm"] else 1)), "flops": 2 * r * c}
    if kind == "quantize":
        return {"bytes": case["rows"] * (4 * case["cols"] + _row_bytes(case["cols"], case["wtype"])),
                "flops": 4 * case["rows"] * case["cols"]}
    dim, _, layers, heads, kv, vocab = SHAPES[case["shape"]]
    kvd = dim // heads * kv
    params = layers * sum(r * c for _, r, c in _shapes(case["shape"]))
    wbytes = layers * sum(r * _row_bytes(c, case["wtype"]) for _, r, c in _shapes(case["shape"]))
    obytes = vocab * _row_bytes(dim, case["wtype"])
    if kind == "decode":
        tokens, outs, seen, kept, passes = 1, 1, case["pos"] + 1, case["pos"] + 1, 1
    elif kind == "prompt":
        n = case["n"]
        tokens, outs, seen, kept, passes = n, 1, n * (n + 1) // 2, 2 * n, 2
    elif kind == "score":
        n = case["n"]
        tokens, outs, seen, kept, passes = n, n, n * (n + 1) // 2, n, 1
    elif kind == "batch":
        seen = int(case["n"] * (0.75 * case["most"] + 1))  # positions are uniform in [most / 2, most]
        tokens, outs, kept, passes = case["n"], case["n"], seen, 1
    else:
        n = case["n"] + 1
        seen = sum(case["pos"] + 1 + i for i in range(n))
        tokens, outs, kept, passes = n, n, seen, n
    return {"bytes": passes * wbytes + (outs if kind == "generate" else 1) * obytes + 8 * layers * kvd * kept + 4 * outs * vocab,
            "flops": 2 * tokens * params + 2 * outs * vocab * dim + 4 * layers * dim * seen}


def tolerance(case):
    return "exact"


# ------------------------------------------------------------------------------------- 64-bit values

def _q8(x):
    """x [.., n] as its Q8_0 blocks give it: scales rounded to fp16, codes to whole numbers."""
    n = x.shape[-1]
    p = torch.nn.functional.pad(x, (0, -n % 32)).unflatten(-1, (-1, 32))
    d = (p.abs().amax(-1, keepdim=True) / 127).half().double()
    c = torch.where(d > 0, torch.round(p / torch.where(d > 0, d, torch.ones_like(d))).clamp(-127, 127), torch.zeros_like(p))
    return (c * d).flatten(-2)[..., :n]


def _norm(x, g):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * g.double()


def _logits(case, seed, toks, want):
    """Logits in 64 bits of the sequences toks [b, n] at the positions that want(b) names, stacked."""
    dim, _, layers, heads, kv, _ = SHAPES[case["shape"]]
    hd, wt = dim // heads, case["wtype"]
    top, lay = _weights(case, seed)
    t = torch.from_numpy(np.asarray(toks, np.int64)).cuda()
    b, n = t.shape
    x = _values(top["tok_embd"][t.flatten()], dim, wt).view(b, n, dim)
    pos = torch.arange(n, device="cuda", dtype=torch.float64)
    ang = pos[:, None] * THETA ** (-2.0 * torch.arange(hd // 2, device="cuda", dtype=torch.float64) / hd)
    cs, sn = torch.cos(ang), torch.sin(ang)
    mask = torch.full((n, n), -math.inf, device="cuda", dtype=torch.float64).triu(1)

    def rope(v):
        v = v.unflatten(-1, (-1, 2))
        e, o = v[..., 0], v[..., 1]
        return torch.stack([e * cs[:, None] - o * sn[:, None], e * sn[:, None] + o * cs[:, None]], -1).flatten(-2)

    def mul(v, name, one):
        rows, cols = sizes[name]
        return _q8(v) @ _values(one[name], cols, wt).T.contiguous()

    sizes = {name: (rows, cols) for name, rows, cols in _shapes(case["shape"])}
    for one in lay:
        h = _norm(x, one["attn_norm"])
        qh = rope(mul(h, "wq", one).view(b, n, heads, hd))
        kh = rope(mul(h, "wk", one).view(b, n, kv, hd)).repeat_interleave(heads // kv, 2)
        vh = mul(h, "wv", one).view(b, n, kv, hd).repeat_interleave(heads // kv, 2)
        att = torch.empty(b, n, heads, hd, device="cuda", dtype=torch.float64)
        for i in range(b):
            for a in range(heads):
                sc = qh[i, :, a] @ kh[i, :, a].T.contiguous() / math.sqrt(hd) + mask
                att[i, :, a] = torch.softmax(sc, -1) @ vh[i, :, a].contiguous()
        x = x + mul(att.flatten(-2), "wo", one)
        h = _norm(x, one["ffn_norm"])
        x = x + mul(torch.nn.functional.silu(mul(h, "w1", one)) * mul(h, "w3", one), "w2", one)
    x = torch.cat([x[i, want(i)] for i in range(b)])
    return _q8(_norm(x, top["norm"])) @ _values(top["output"], dim, wt).T.contiguous()


def exact(case, seed):
    kind = case["kind"]
    if kind == "decode":
        return _logits(case, seed, _tokens(case, seed, case["pos"] + 1)[None], lambda i: [case["pos"]])[0]
    if kind == "prompt":
        return _logits(case, seed, _tokens(case, seed, case["n"])[None], lambda i: [case["n"] - 1])[0]
    if kind == "score":
        return _logits(case, seed, _tokens(case, seed, case["n"])[None], lambda i: list(range(case["n"])))
    if kind == "batch":
        toks, pos = _batch_state(case, seed)
        rows = [_logits(case, seed, toks[i:i + 16], lambda j, i=i: [int(pos[i + j])]) for i in range(0, case["n"], 16)]
        return torch.cat(rows)
    if kind == "generate":
        return None  # which tokens are drawn turns on the last bits of the probabilities
    g = _gen(seed, 2)
    if kind == "matmul":
        a = torch.randn(case["m"], case["k"], device="cuda", generator=g).double()
        b = torch.randn(case["n"], case["k"], device="cuda", generator=g).double()
        return a @ b.T.contiguous()
    if kind == "matvec":
        raw, x, gain = _matvec_inputs(case, g)
        x = x.double()
        if gain is not None:
            x = _norm(x, gain)
        if case["wtype"] != "f32":
            x = _q8(x)
        return _values(raw, case["cols"], case["wtype"]) @ x
    return None  # bytes
