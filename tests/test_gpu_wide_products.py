"""Products of 17 to 64 rows and more than a thousand strips: three and four strips a block with a last block that is not full, and a strip of fewer columns,
against 64 bits; weights past the caches the same bits."""
import numpy as np
import pytest

from test_gpu_mid_products import setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K", [(16 * 1025 + 3, 96), (16 * 1535, 544), (16 * 1537 + 9, 288), (16 * 2047, 32)])
@pytest.mark.parametrize("M", [17, 33, 48, 49, 64])
def test_wide(N, K, M):
    rt, k, A, S, ws, z = setup(N, K, N, N + M)
    want, seen = 30.0 * np.tanh(z[:M] / 30.0), []
    for once in (1, 3):
        C = rt.upload(np.full((M + 1, N + 5), 3.0, np.float32))
        k.zk_gemm_bf16(A.ptr, K, S.ptr, C.ptr, N + 5, 1, M, N, K, 1, 30.0, once, ws.ptr, ws.nbytes, None, rt.stream)
        got = rt.download(C)
        # float sums of K products of size K^-0.5, and the float tanh
        assert np.abs(got[:M, :N] - want).max() < 2e-5 * np.abs(want).max()
        assert (got[M:] == 3.0).all() and (got[:, N:] == 3.0).all()
        seen.append(got)
    assert np.array_equal(*seen)
