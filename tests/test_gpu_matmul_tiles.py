"""qmh_matmul_nt (k_gemm_nt) at the edges of its 16 x 16 tiles, 16-value groups and 256-value panels, with
unaligned rows and special values, against the oracle: bits (a NaN as a NaN)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,off", [(1, 1, 3, 0), (15, 17, 16, 0), (16, 16, 15, 1), (33, 31, 47, 3), (32, 48, 256, 0),
                                       (17, 65, 257, 2), (1, 130, 511, 0), (70, 5, 513, 1), (47, 33, 784, 0)])
def test_tile_edges(gpu, oracle, M, N, K, off):
    print("case", M, N, K, off, flush=True)
    rs = np.random.default_rng(M * N + K)
    A = rs.standard_normal((M, K)).astype(np.float32)
    B = rs.standard_normal((N, K)).astype(np.float32)
    A[0, 0], B[0, K - 1], A[M - 1, K // 2], B[N - 1, 0] = -0.0, 1e-41, 3e38, np.inf
    if M > 2:
        A[1, K - 1] = np.nan
    L = gpu.load_library()
    a, b = gpu.DeviceBuffer(4 * (M * K + off)), gpu.DeviceBuffer(4 * (N * K + off))
    c = gpu.DeviceBuffer(4 * M * N)
    for d, x in ((a, A), (b, B)):
        assert L.qmh_memcpy_h2d(d.ptr + 4 * off, x.ctypes.data, x.nbytes) == 0
    assert L.qmh_matmul_nt(a.ptr + 4 * off, b.ptr + 4 * off, c.ptr, M, N, K, None) == 0
    got, want = c.to_array(np.float32).reshape(M, N), oracle.gemm_nt(A, B)
    nan = np.isnan(want)
    assert np.array_equal(nan, np.isnan(got))
    assert np.array_equal(got.view(np.uint32)[~nan], want.view(np.uint32)[~nan])


def sweep(rs, n):
    """n values over every exponent, subnormal ones among them, with ties at the last subnormal bit"""
    v = np.ldexp(rs.uniform(1, 2, n), rs.integers(-149, 128, n)).astype(np.float32)
    k = n // 8
    v[:k] = np.ldexp(rs.integers(1, 1 << 12, k).astype(np.float64), -149)  # few bits: halves of them tie
    v[k:2 * k] = np.ldexp(1.0, rs.integers(-40, 1, k))
    v[2 * k:3 * k] = np.ldexp(rs.uniform(1, 2, k), rs.integers(-80, -60, k))  # products around 2^-149
    v[3 * k:3 * k + 4] = [0.0, np.inf, np.nan, np.float32(3.4028235e38)]
    rs.shuffle(v)
    return v * rs.choice([-1, 1], n).astype(np.float32)


# products alone (K = 1) and chains of a few, where subnormal inputs, products and sums decide the bits: flushing
# any of them to zero, or rounding a product twice, shows
@pytest.mark.parametrize("K", [1, 2, 5])
def test_every_exponent(gpu, oracle, K):
    print("case", K, flush=True)
    rs = np.random.default_rng(K)
    A, B = sweep(rs, 512 * K).reshape(512, K), sweep(rs, 512 * K).reshape(512, K)
    want = oracle.gemm_nt(A, B)
    tiny = np.abs(want) < np.float32(2.0 ** -126)
    assert (tiny & (want != 0)).mean() > (0.02 if K == 1 else 0.002)  # the oracle's results do hold subnormals
    c = gpu.DeviceBuffer(4 * want.size)
    a, b = gpu.DeviceBuffer.from_array(A), gpu.DeviceBuffer.from_array(B)
    assert gpu.load_library().qmh_matmul_nt(a.ptr, b.ptr, c.ptr, 512, 512, K, None) == 0
    got = c.to_array(np.float32).reshape(512, 512)
    nan = np.isnan(want)
    assert np.array_equal(nan, np.isnan(got))
    assert np.array_equal(got.view(np.uint32)[~nan], want.view(np.uint32)[~nan])
