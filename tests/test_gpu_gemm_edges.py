"""Tile products whose last row of tiles is not full: the rows of C, and nothing behind them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [65, 127, 129, 191, 257, 535, 769])      # around 64, 128 and 256 rows
@pytest.mark.parametrize("N,K,gated", [(256, 64, 0), (384, 2304, 0), (4608, 512, 0), (9216, 128, 1), (144, 256, 1)])
def test_rows(M, N, K, gated):
    from zse_amd.runtime.device import Runtime
    from zse_amd.weights.safetensors import bf16_bits_to_f32, f32_to_bf16_bits
    rt = Runtime.get()
    k = rt.kernels("bfloat16")
    rng = np.random.default_rng(M + N)
    bits = lambda *shape: f32_to_bf16_bits(rng.normal(size=shape).astype(np.float32) * K ** -0.25)
    a, w = bits(M, K), bits(N * (1 + gated), K)
    A, W, C = rt.upload(a, "bfloat16"), rt.upload(w, "bfloat16"), rt.upload(np.full((M + 3, N + 8), 0x4040, np.uint16), "bfloat16")
    S = rt.empty(w.shape, "bfloat16")
    k.zk_strip_layout(W.ptr, S.ptr, *w.shape, rt.stream)
    ws = rt.zeros((k.zk_gemm_bf16_workspace() // 4,), "float32")
    k.zk_gemm_bf16(A.ptr, K, S.ptr, C.ptr, N + 8, 0, M, N, K, 5 if gated else 0, 0.0, 1, ws.ptr, ws.nbytes, None, rt.stream)
    got = rt.download_f32(C)
    want = bf16_bits_to_f32(a).astype(np.float64) @ bf16_bits_to_f32(w).astype(np.float64).T
    if gated:
        want = np.maximum(want[:, :N], 0) * want[:, N:]
    # a result rounded to 8 bits of mantissa; K float additions of products of size K^-0.5
    assert (np.abs(got[:M, :N] - want) <= np.abs(want) * 2.0 ** -8 + 1e-4 * (1 + 3 * gated)).all()
    assert (got[M:] == 3.0).all() and (got[:, N:] == 3.0).all()
