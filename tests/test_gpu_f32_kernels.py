"""The 32-bit path's matrix-core kernels at the edges of their tiles, against 64-bit arithmetic."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    from zse_amd.runtime.device import Runtime
    return Runtime.get()


# rows around 16 and 64 and many of them; columns around 16, 32 and 64; K below a step, around the
# eight waves' steps of 32, odd (values loaded one by one) and with rows further apart than K
@pytest.mark.parametrize("M,N,K,gap", [(1, 16, 4, 0), (3, 33, 31, 0), (16, 1000, 256, 4), (17, 64, 260, 0), (15, 16400, 64, 0),
                                       (63, 65, 1024, 0), (64, 64, 36, 8), (300, 4096, 1028, 0), (129, 8200, 100, 3), (5, 7, 1, 0)])
def test_product(rt, M, N, K, gap):
    k = rt.kernels("float32")
    rng = np.random.default_rng(M + N + K)
    a, w = rng.normal(size=(M, K + gap)).astype(np.float32), rng.normal(size=(N, K)).astype(np.float32)
    A, W = rt.upload(a), rt.upload(w)
    C, one = rt.upload(np.full((M, N + 3), 7.0, np.float32)), rt.empty((1, N), "float32")
    k.zk_gemm_plain(A.ptr, K + gap, W.ptr, C.ptr, N + 3, 1, M, N, K, rt.stream)
    got = rt.download(C)
    want = a[:, :K].astype(np.float64) @ w.astype(np.float64).T
    # K roundings of partial sums of at most sqrt(K) size, 2^-24 each, and a margin of 8 for the largest of the values
    assert np.abs(got[:, :N] - want).max() < 8 * 2.0 ** -24 * max(K, 8)
    assert (got[:, N:] == 7.0).all()
    for m in {0, M // 2, M - 1}:        # a row's bits do not depend on the rows beside it
        k.zk_gemm_plain(A.ptr + 4 * m * (K + gap), K + gap, W.ptr, one.ptr, N, 1, 1, N, K, rt.stream)
        assert np.array_equal(rt.download(one)[0], got[m, :N]), m
