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
