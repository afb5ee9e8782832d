"""32-bit products by tiles of 64 x 32 and 80 x 64: rows and columns that do not fill a tile, K not in whole steps or pieces; a row's bits are those
of the row alone (by the tiles of up to sixteen rows)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 64 x 32: one round of 255 and 256 blocks; 80 x 64: a round that the larger tile fills, the smaller exceed
@pytest.mark.parametrize("M,N", [(64, 8192), (57, 8150), (150, 8192), (143, 8129), (303, 8192)])
@pytest.mark.parametrize("K", [512, 1024, 514, 1023, 548])
def test_tiles(M, N, K):
    from zse_amd.runtime.device import Runtime
    rt = Runtime.get()
    k = rt.kernels("float32")
    rng = np.random.default_rng(M + N + K)
    a, w = rng.standard_normal((M, K), dtype=np.float32), rng.standard_normal((N, K), dtype=np.float32) * np.float32(K ** -0.5)
    A, W = rt.upload(a), rt.upload(w)
    C = rt.upload(np.full((M + 1, N + 3), 3.0, np.float32))
    k.zk_gemm_plain(A.ptr, K, W.ptr, C.ptr, N + 3, 1, M, N, K, rt.stream)
    got = rt.download(C)
    want = a.astype(np.float64) @ w.astype(np.float64).T
    # float sums of K products of size K^-0.5
    assert np.abs(got[:M, :N] - want).max() < 3e-6 * np.abs(want).max()
    assert (got[M:] == 3.0).all() and (got[:, N:] == 3.0).all()
    one = rt.zeros((1, N), "float32")
    for m in (0, M // 2, M - 1):
        k.zk_gemm_plain(A.ptr + m * K * 4, K, W.ptr, one.ptr, N, 1, 1, N, K, rt.stream)
        assert np.array_equal(rt.download(one)[0], got[m, :N]), m
