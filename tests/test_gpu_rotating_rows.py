"""The rotating product of 17 to 64 rows against the product and the rotation as launches of their own: results that differ by the order of
the product's sums alone, and nothing stored for a row without a slot."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# one strip a block (up to 256 strips) and two, the last block not full; chunks that K does not fill; no keys of its own; both layouts of values
@pytest.mark.parametrize("nh,nkv,hd,K,vt", [(8, 4, 256, 2304, 1), (3, 1, 16, 96, 0), (2, 1, 80, 288, 1), (32, 16, 128, 512, 1), (4, 0, 64, 1024, 1),
                                            (33, 15, 96, 160, 0)])
@pytest.mark.parametrize("M", [17, 32, 33, 48, 64])
def test_rows(M, nh, nkv, hd, K, vt):
    from zse_amd.runtime.device import Runtime
    from zse_amd.weights.safetensors import f32_to_bf16_bits
    rt = Runtime.get()
    k = rt.kernels("bfloat16")
    rng = np.random.default_rng(M + hd + K)
    N, bs, pages = (nh + 2 * nkv) * hd, 8, 12
    up = lambda x: rt.upload(f32_to_bf16_bits(np.ascontiguousarray(x, np.float32)), "bfloat16")
    A, W, S = up(rng.normal(size=(M, K))), up(rng.normal(size=(N, K)) * K ** -0.5), rt.empty((N, K), "bfloat16")
    k.zk_strip_layout(W.ptr, S.ptr, N, K, rt.stream)
    pos = rt.upload(rng.integers(0, 8000, M).astype(np.int32))
    slot = rng.permutation(pages * bs)[:M].astype(np.int32)
    slot[M // 3] = -1
    slots = rt.upload(slot)
    freq = rt.upload((10000.0 ** (-np.arange(hd // 2) * 2 / hd)).astype(np.float32))
    assert k.zk_qkv_rope_rows_bf16_supports(M, K, hd, hd)
    assert not any(k.zk_qkv_rope_rows_bf16_supports(*a) for a in ((16, K, hd, hd), (65, K, hd, hd), (M, K, hd, hd // 2), (M, K + 8, hd, hd)))
    ws = rt.zeros((k.zk_gemm_bf16_workspace() // 4,), "float32")
    res = []
    for own in (1, 0):
        Q = rt.zeros((M, N), "bfloat16")
        kc, vc = (rt.zeros((pages * bs * max(nkv, 1) * hd,), "bfloat16") for _ in range(2))
        sl = slots.ptr if nkv else None
        if own:
            k.zk_qkv_rope_rows_bf16(A.ptr, K, S.ptr, Q.ptr, N, M, K, 3, pos.ptr, sl, freq.ptr, kc.ptr, vc.ptr, nh, nkv, hd, bs, vt, rt.stream)
        else:
            k.zk_gemm_bf16(A.ptr, K, S.ptr, Q.ptr, N, 0, M, N, K, 0, 0.0, 1, ws.ptr, ws.nbytes, None, rt.stream)
            k.zk_rope_cache_write(Q.ptr, pos.ptr, sl, freq.ptr, hd, kc.ptr, vc.ptr, M, nh, nkv, hd, bs, vt, rt.stream)
        res.append([rt.download_f32(t) for t in (Q, kc, vc)])
    for i, (a, b) in enumerate(zip(*res)):
        if i == 0:
            a, b = a[:, :nh * hd], b[:, :nh * hd]
        # a value rounded to 8 bits of mantissa may round the other way, before it is turned and after, and its partner too
        assert np.abs(a - b).max() <= 3 * 2.0 ** -8 * np.abs(b).max()
        assert np.mean(a != b) < 0.02
        assert np.array_equal(a == 0, b == 0)
