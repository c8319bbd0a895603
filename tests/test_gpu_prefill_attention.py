"""The prompt attention kernels (scores, softmax, P.V of P tokens at once) called by themselves, against a
float32 restatement in the reference's order of operations with the oracle's softmax: bits, no
tolerance. Positions and tokens sit at the edges of the tiles (16 and 64 tokens, 64 positions, 8 positions
per load), the row lengths at the edges of the softmax's instances (128, 256, 512, 1024, 2048, 4096)."""
import ctypes

import numpy as np
import pytest

from _boundary import softmax_boundary_input

pytestmark = pytest.mark.gpu


def run(gpu, q, kt, v, P, pos0, n_heads, n_kv, hd, S, scale, image=None, skew=0):
    """out, or with image (perm8: 0 or 1) its quantized codes and scales; the queries skew bytes past alignment, kt and
    v arrays or device buffers"""
    L = gpu.load_library()
    fn = L.qmh_launch_pf_attention
    fn.restype = ctypes.c_int
    vp, i32 = ctypes.c_void_p, ctypes.c_int
    fn.argtypes = [vp] * 5 + [i32] * 6 + [ctypes.c_float, vp, vp, i32, i32, vp]
    b = [gpu.DeviceBuffer(q.nbytes + skew)] + [gpu.DeviceBuffer.from_array(a) for a in (kt, v) if isinstance(a, np.ndarray)]
    dk, dv = b[1:] or (kt, v)
    att, out = gpu.DeviceBuffer(n_heads * P * S * 4), gpu.DeviceBuffer(P * n_heads * hd * 4)
    PP = 128
    xc, xd = gpu.DeviceBuffer(PP * n_heads * hd), gpu.DeviceBuffer(PP * n_heads * hd // 32 * 4)
    try:
        assert L.qmh_memcpy_h2d(b[0].ptr + skew, q.ctypes.data, q.nbytes) == 0
        for x in (att, out, xc, xd):
            assert L.qmh_memset(x.ptr, 0xff, x.nbytes) == 0  # NaN wherever nothing is written
        rc = fn(b[0].ptr + skew, dk.ptr, dv.ptr, att.ptr, out.ptr, P, pos0, n_heads, n_kv, hd, S, float(scale),
                None if image is None else xc.ptr, None if image is None else xd.ptr, PP, image or 0, L.qmh_stream())
        assert rc == 0
        gpu.sync()
        if image is None:
            return out.to_array(np.float32).reshape(P, n_heads, hd)
        codes = xc.to_array(np.int8).reshape(-1, PP, 32)[:, :P]
        return codes, xd.to_array(np.float32).reshape(-1, PP)[:, :P]
    finally:
        for x in b + [att, out, xc, xd]:
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
    q[0, 0, :4] = [0.0, -0.0, 1e-40, 3e38]  # signed zeros, a subnormal, products that overflow
    kt[:4, 0] = [-1.0, 1.0, 1e-3, 0.25]
    v[pos0 + P:] = np.nan  # positions nobody sees
    v[0, 0], v[min(1, S - 1), 1] = -0.0, 1e-41
    scale = 1.0 / np.sqrt(np.float32(hd))
    got = run(gpu, q, kt, v, P, pos0, n_heads, n_kv, hd, S, scale)
    ref = want(oracle, q, kt, v, P, pos0, n_heads, n_kv, hd, scale)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), np.argwhere(got.view(np.uint32) != ref.view(np.uint32))[:5]


# scores and P.V whose products and sums are all subnormal: score chains below 2^-126, which the scale brings to the
# order of one, and values of V below 2^-126. A product or a sum flushed to zero would change every output.
@pytest.mark.parametrize("hd,n_heads,n_kv,P,pos0", [(48, 2, 1, 18, 0), (64, 2, 2, 33, 70), (128, 2, 1, 17, 130)])
def test_subnormal_chains(gpu, oracle, hd, n_heads, n_kv, P, pos0):
    print("case", hd, n_heads, n_kv, P, pos0, flush=True)
    rs = np.random.default_rng(hd)
    S = pos0 + P
    q = (rs.standard_normal((P, n_heads, hd)) * 2.0 ** -66).astype(np.float32)
    kt = (rs.standard_normal((n_kv * hd, S)) * 2.0 ** -66).astype(np.float32)
    v = (rs.standard_normal((S, n_kv * hd)) * 2.0 ** -129).astype(np.float32)
    scale = np.float32(2.0 ** 127)
    chains = np.einsum("phd,hdt->pht", q.astype(np.float64), np.stack([kt[h // (n_heads // n_kv) * hd:][:hd]
                                                                       for h in range(n_heads)]).astype(np.float64))
    assert np.abs(chains).max() < 2.0 ** -126 and np.abs(chains * float(scale)).max() > 0.1
    ref = want(oracle, q, kt, v, P, pos0, n_heads, n_kv, hd, scale)
    assert 0 < np.abs(ref).max() < 2.0 ** -126
    got = run(gpu, q, kt, v, P, pos0, n_heads, n_kv, hd, S, scale)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))


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


# the quantized image from the general kernels, where the queries' alignment keeps the others out: the same
# codes and scales, both byte orders
@pytest.mark.parametrize("hd,n_heads,n_kv,P,pos0,S", [(64, 2, 1, 19, 3, 64), (128, 2, 2, 5, 300, 310)])
@pytest.mark.parametrize("perm8", [0, 1])
def test_image_of_unaligned_queries(gpu, hd, n_heads, n_kv, P, pos0, S, perm8):
    print("case", hd, n_heads, n_kv, P, pos0, S, perm8, flush=True)
    rs = np.random.default_rng(hd + P)
    q = rs.standard_normal((P, n_heads, hd)).astype(np.float32)
    kt = rs.standard_normal((n_kv * hd, S)).astype(np.float32)
    v = rs.standard_normal((S, n_kv * hd)).astype(np.float32)
    a = run(gpu, q, kt, v, P, pos0, n_heads, n_kv, hd, S, hd ** -0.5, image=perm8)
    b = run(gpu, q, kt, v, P, pos0, n_heads, n_kv, hd, S, hd ** -0.5, image=perm8, skew=4)
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1].view(np.uint32), b[1].view(np.uint32))


# a layer's keys and values past 2 GiB (the MFMA kernels' 32-bit offsets) and past 4 GiB (the general kernels): 64
# heads x 64 dimensions, a token at the end of S positions, random values in the first and last heads' keys and in
# the first and last 64 positions' V (zeros elsewhere), the probabilities of every position. Then the same token's
# image, from aligned and unaligned queries.
@pytest.mark.parametrize("S", [262000, 262208])
def test_large_caches(gpu, oracle, S):
    print("case", S, flush=True)
    nh, hd, n = 64, 64, 64
    L = gpu.load_library()
    rs = np.random.default_rng(9)
    q = rs.standard_normal((1, nh, hd)).astype(np.float32)
    k = {h: 0.1 * rs.standard_normal((hd, S)).astype(np.float32) for h in (0, nh - 1)}
    v = {t: rs.standard_normal((n, nh * hd)).astype(np.float32) for t in (0, S - n)}
    dk, dv = gpu.DeviceBuffer(4 * nh * hd * S), gpu.DeviceBuffer(4 * nh * hd * S)
    try:
        for d in (dk, dv):
            assert L.qmh_memset(d.ptr, 0, d.nbytes) == 0
        for h, x in k.items():
            assert L.qmh_memcpy_h2d(dk.ptr + 4 * h * hd * S, x.ctypes.data, x.nbytes) == 0
        for t, x in v.items():
            assert L.qmh_memcpy_h2d(dv.ptr + 4 * t * nh * hd, x.ctypes.data, x.nbytes) == 0
        scale = np.float32(hd ** -0.5)
        got = run(gpu, q, dk, dv, 1, S - 1, nh, nh, hd, S, scale)
        images = [run(gpu, q, dk, dv, 1, S - 1, nh, nh, hd, S, scale, image=1, skew=s) for s in (0, 4)]
    finally:
        dk.free()
        dv.free()
    for h in k:
        s = np.zeros(S, np.float32)
        for d in range(hd):
            s = s + q[0, h, d] * k[h][d]
        pr = oracle.softmax(s * scale)
        acc = np.zeros(hd, np.float32)  # zeros of V add +0 to a chain from +0
        for t0, x in v.items():
            for t in range(n):
                acc = acc + pr[t0 + t] * x[t, h * hd:(h + 1) * hd]
        assert np.array_equal(got[0, h].view(np.uint32), acc.view(np.uint32)), h
    assert np.array_equal(images[0][0], images[1][0])
    assert np.array_equal(images[0][1].view(np.uint32), images[1][1].view(np.uint32))
