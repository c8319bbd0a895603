"""The tiled prefill matmul (k_pf_gemm) at the edges of its tiles, against the one-token-at-a-time path on
the same model (itself held to the oracle by test_gpu_model.py). Comparisons are of bits: both paths
take every sum in the reference's order, so no tolerance applies; a NaN is compared as a NaN."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def blocks(rng, rows, cols, wt, small=0.0):
    """rows of Q8_0 / Q4_0 blocks with random codes and scales (a share `small` of them subnormal fp16)."""
    nb, cb = (cols + 31) // 32, 32 if wt == "q8_0" else 16
    b = rng.integers(0, 256, (rows, nb, 2 + cb), np.uint8)
    if wt == "q8_0":
        b[:, :, 2:][b[:, :, 2:] == 128] = 7
    d = (rng.uniform(0.2, 1.0, (rows, nb)) * (2e-4 if wt == "q8_0" else 4e-3)).astype(np.float16)
    tiny = rng.random((rows, nb)) < small
    d[tiny] = rng.integers(1, 1024, int(tiny.sum())).astype(np.uint16).view(np.float16)
    b[:, :, :2] = d.view(np.uint8).reshape(rows, nb, 2)
    pad = nb * 32 - cols  # values past the row are zero in a real file
    if pad and wt == "q8_0":
        b[:, -1, 2 + 32 - pad:] = 0
    elif pad:
        v = np.stack([b[:, -1, 2:] & 15, b[:, -1, 2:] >> 4], 2).reshape(rows, 32)
        v[:, 32 - pad:] = 8
        b[:, -1, 2:] = v[:, 0::2] | v[:, 1::2] << 4
    return np.ascontiguousarray(b.reshape(rows, -1))


def model(gpu, dim, hidden, heads, kv, vocab, max_seq, wt, edit=None, seed=5):
    rng = np.random.default_rng(seed)
    kvd = dim // heads * kv
    sizes = {"wq": (dim, dim), "wk": (kvd, dim), "wv": (kvd, dim), "wo": (dim, dim), "w1": (hidden, dim),
             "w2": (dim, hidden), "w3": (hidden, dim), "tok_embd": (vocab, dim), "output": (vocab, dim)}
    t = {n: blocks(rng, r, c, wt, 0.02) for n, (r, c) in sizes.items()}
    for n in ("attn_norm", "ffn_norm", "norm"):
        t[n] = (1 + 0.1 * rng.standard_normal(dim)).astype(np.float32)
    if edit:
        edit(t)

    def view(name):
        v = gpu.TensorView()
        v.data = t[name].ctypes.data
        if name in sizes:
            v.dtype, v.ndim, (v.ne[0], v.ne[1]) = gpu.DTYPES[wt], 2, sizes[name]
        else:
            v.dtype, v.ndim, v.ne[0] = gpu.F32, 1, dim
        return v

    layer = (gpu.TensorView * 9)(*[view(n) for n in ("attn_norm", "wq", "wk", "wv", "wo", "ffn_norm", "w1", "w2", "w3")])
    cfg = gpu.QmhConfig(dim, hidden, 1, heads, kv, vocab, max_seq, 10000.0, 1e-5)
    e, n, o = view("tok_embd"), view("norm"), view("output")
    h = gpu.load_library().qmh_model_create(ctypes.byref(cfg), ctypes.byref(e), ctypes.byref(n), ctypes.byref(o), layer)
    assert h, gpu.last_error()
    return gpu.Model(h)


def same(a, b):
    na, nb = np.isnan(a), np.isnan(b)
    return np.array_equal(na, nb) and np.array_equal(a.view(np.uint32)[~na], b.view(np.uint32)[~na])


def check(m, monkeypatch, P, vocab):
    rng = np.random.default_rng(P)
    toks = rng.integers(0, vocab, P).astype(np.int32)
    got = m.prefill(toks, 0, want_logits=True)
    tail = m.forward(3, P).copy()
    monkeypatch.setenv("QMH_PREFILL_SEQ", "1")
    want = m.prefill(toks, 0, want_logits=True)
    assert same(got, want), np.argwhere(got.view(np.uint32) != want.view(np.uint32))[:5]
    assert same(tail, m.forward(3, P))


# tokens around the 32- and 64-token tiles; rows that end inside a 32-row tile and a workgroup; 3, 9 and 11
# blocks per row (whole and partial stages of 4, partial last blocks). The 20001-row output takes the
# 4 x 2 workgroups, the others the 2 x 2 ones.
@pytest.mark.parametrize("wt", ["q4_0", "q8_0"])
@pytest.mark.parametrize("dim,hidden,vocab,P", [(72, 200, 300, 65), (72, 344, 20001, 96), (288, 330, 517, 97),
                                                (64, 32, 90, 128), (72, 200, 20001, 191), (288, 768, 300, 129)])
def test_tile_edges(gpu, monkeypatch, dim, hidden, vocab, P, wt):
    print(f"case {dim} {hidden} {vocab} {P} {wt}", flush=True)
    with model(gpu, dim, hidden, 6 if dim % 6 == 0 else 4, 2, vocab, 256, wt) as m:
        check(m, monkeypatch, P, vocab)


# infinite and NaN weight scales: only the rows that hold them change
@pytest.mark.parametrize("wt", ["q4_0", "q8_0"])
@pytest.mark.parametrize("where,vocab", [("output", 300), ("output", 20001), ("w1", 300)])
def test_nonfinite_scales(gpu, monkeypatch, where, vocab, wt):
    print(f"case {where} {vocab} {wt}", flush=True)
    bs = 34 if wt == "q8_0" else 18

    def edit(t):
        b = t[where].reshape(t[where].shape[0], -1, bs)
        for row, blk, half in ((0, 1, 0x7c00), (5, 0, 0x7e00), (37, 2, 0xfc00), (199, 1, 0x7c00)):
            b[row, blk, :2] = np.array([half], np.uint16).view(np.uint8)

    with model(gpu, 72, 200, 6, 2, vocab, 256, wt, edit) as m:
        check(m, monkeypatch, 70, vocab)


# both sides of the rule that takes 8 to 64 tokens to the tiled matmul (300000 rows x tokens up to 32 tokens), for
# the output (row counts that end inside tiles) and for W1 | W3, whose input image to W2 changes with it; one and
# two token tiles
@pytest.mark.parametrize("wt", ["q4_0", "q8_0"])
@pytest.mark.parametrize("hidden,vocab,P", [(200, 37501, 7), (200, 37500, 8), (200, 37499, 8), (200, 9376, 32),
                                            (200, 9376, 31), (200, 9091, 33), (4688, 300, 32), (4687, 300, 32),
                                            (2381, 300, 63), (2380, 300, 63), (2344, 4688, 64)])
def test_few_token_rule(gpu, monkeypatch, hidden, vocab, P, wt):
    print(f"case {hidden} {vocab} {P} {wt}", flush=True)
    with model(gpu, 72, hidden, 6, 2, vocab, 128, wt) as m:
        check(m, monkeypatch, P, vocab)


# the same from 33 tokens on, where the line depends on the columns: below 8 blocks (1000000; W1 | W3 400000), below
# 16 (450000), from 16 on (300000)
@pytest.mark.parametrize("dim,hidden,vocab,P", [(72, 200, 15625, 64), (72, 200, 15624, 64), (72, 3125, 300, 64),
                                                (72, 3124, 300, 64), (288, 32, 7032, 64), (288, 32, 7031, 64),
                                                (288, 6061, 300, 33), (288, 6060, 300, 33), (528, 32, 4688, 64),
                                                (528, 32, 4687, 64)])
def test_few_token_rule_by_columns(gpu, monkeypatch, dim, hidden, vocab, P):
    print(f"case {dim} {hidden} {vocab} {P}", flush=True)
    with model(gpu, dim, hidden, 6, 2, vocab, 128, "q4_0") as m:
        check(m, monkeypatch, P, vocab)
