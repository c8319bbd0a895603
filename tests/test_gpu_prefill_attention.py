"""The prompt attention kernels (scores, softmax, P.V of P tokens at once) called by themselves, against a
float32 restatement in the reference's order of operations with the oracle's softmax: bits, no
tolerance. Positions and tokens sit at the edges of the tiles (16 and 64 tokens, 64 positions, 8 positions
per load), the row lengths at the edges of the softmax's instances (128, 256, 512, 1024, 2048, 4096)."""
import ctypes

import numpy as np
import pytest

from _boundary import softmax_boundary_input

pytestmark = pytest.mark.gpu


def run(gpu, q, kt, v, P, pos0, n_heads, n_kv, hd, S, scale):
    L = gpu.load_library()
    fn = L.qmh_launch_pf_attention
    fn.restype = ctypes.c_int
    vp, i32 = ctypes.c_void_p, ctypes.c_int
    fn.argtypes = [vp] * 5 + [i32] * 6 + [ctypes.c_float, vp, vp, i32, i32, vp]
    b = [gpu.DeviceBuffer.from_array(a) for a in (q, kt, v)]
    att, out = gpu.DeviceBuffer(n_heads * P * S * 4), gpu.DeviceBuffer(P * n_heads * hd * 4)
    try:
        assert gpu.load_library().qmh_memset(att.ptr, 0xff, att.nbytes) == 0  # NaN wherever nothing is written
        rc = fn(b[0].ptr, b[1].ptr, b[2].ptr, att.ptr, out.ptr, P, pos0, n_heads, n_kv, hd, S, float(scale), None, None,
                128, 0, L.qmh_stream())
        assert rc == 0
        gpu.sync()
        return out.to_array(np.float32).reshape(P, n_heads, hd)
    finally:
        for x in b + [att, out]:
            x.free()


def want(oracle, q, kt, v, P, pos0, n_heads, n_kv, hd, scale):
    out = np.zeros((P, n_heads, hd), np.float32)
    for h in range(n_heads):
        k = h // (n_heads // n_kv)
        s = np.zeros((P, pos0 + P), np.float32)
        for d in range(hd):
            s = s + q[:, h, d][:, None] * kt[k * hd + d, :pos0 + P][None]
        s = s * np.float32(scale)
        for p in range(P):
            pr = oracle.softmax(s[p, :pos0 + p + 1].copy())
            acc = np.zeros(hd, np.float32)
            for t in range(pos0 + p + 1):
                acc = acc + pr[t] * v[t, k * hd:(k + 1) * hd]
            out[p, h] = acc
    return out


@pytest.mark.parametrize("hd,n_heads,n_kv,P,pos0,S", [
    (48, 2, 1, 67, 0, 67), (48, 2, 2, 18, 61, 80), (64, 2, 1, 33, 0, 33), (64, 2, 2, 17, 239, 257),
    (128, 1, 1, 16, 0, 16), (128, 2, 1, 15, 499, 515), (128, 1, 1, 3, 1021, 1027), (64, 1, 1, 5, 2044, 2049),
    (64, 1, 1, 2, 4095, 4097), (32, 2, 2, 19, 100, 121),
    # contexts that end at max_seq: the last 4-position loads run past the last row, the sets loaded ahead past V
    (64, 1, 1, 1, 0, 1), (64, 2, 1, 1, 5, 6), (128, 2, 2, 2, 9, 11), (48, 2, 1, 17, 6, 23), (128, 1, 1, 16, 493, 509)])
def test_against_restatement(gpu, oracle, hd, n_heads, n_kv, P, pos0, S):
    print("case", hd, n_heads, n_kv, P, pos0, S, flush=True)
    rs = np.random.default_rng(hd + P + pos0)
    q = rs.standard_normal((P, n_heads, hd)).astype(np.float32)
    kt = rs.standard_normal((n_kv * hd, S)).astype(np.float32)
    v = rs.standard_normal((S, n_kv * hd)).astype(np.float32)
    q[0, 0, :4] = [0.0, -0.0, 1e-40, 3e38]  # signed zeros, a subnormal, a product that overflows
    kt[:4, 0] = [-1.0, 1.0, 1e-3, 0.25]
    v[pos0 + P:] = np.nan  # positions nobody sees
    v[0, 0], v[min(1, S - 1), 1] = -0.0, 1e-41
    scale = 1.0 / np.sqrt(np.float32(hd))
    got = run(gpu, q, kt, v, P, pos0, n_heads, n_kv, hd, S, scale)
    ref = want(oracle, q, kt, v, P, pos0, n_heads, n_kv, hd, scale)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), np.argwhere(got.view(np.uint32) != ref.view(np.uint32))[:5]


# rows whose sum of exponentials sits on a float midpoint of its reciprocal: the tree sum cannot decide it,
# and the reference's serial sum is taken. Scores are given exactly (query 1, 0, 0, ..; key row 0 the score).
@pytest.mark.parametrize("n", [90, 200, 300, 500, 700, 1500, 3000])
def test_serial_sum(gpu, oracle, n):
    print("case", n, flush=True)
    hd = 64
    for seed in range(4):
        s = softmax_boundary_input(n, seed)
        q = np.zeros((1, 1, hd), np.float32)
        q[0, 0, 0] = 1.0
        kt = np.zeros((hd, n), np.float32)
        kt[0] = s
        v = np.zeros((n, hd), np.float32)
        idx = np.argsort(-s)[:hd]  # column i reads the probability of the i-th largest score
        v[idx, np.arange(hd)] = 1.0
        got = run(gpu, q, kt, v, 1, n - 1, 1, 1, hd, n, 1.0)
        assert np.array_equal(got[0, 0].view(np.uint32), oracle.softmax(s)[idx].view(np.uint32)), (n, seed)
