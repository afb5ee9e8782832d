"""Decoded tokens' values past the caches: the same bits as through them, by both kernels, over the pages that take it and those that do not."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh,nkv,hd,vd", [(8, 4, 256, 256), (4, 2, 128, 128), (4, 4, 64, 64), (4, 2, 32, 32), (4, 4, 128, 64)])
@pytest.mark.parametrize("bs", [4, 8, 16, 32, 64])
@pytest.mark.parametrize("long_table", [False, True])
def test_bits(nh, nkv, hd, vd, bs, long_table):
    from zse_amd.runtime.device import Runtime
    from zse_amd.weights.safetensors import f32_to_bf16_bits
    rt = Runtime.get()
    k = rt.kernels("bfloat16")
    rng = np.random.default_rng(hd + bs)
    up = lambda *shape: rt.upload(f32_to_bf16_bits(rng.standard_normal(shape, dtype=np.float32)), "bfloat16")
    lens = [1, 33, 128, 300, 513]
    R, need = len(lens), [-(-n // bs) for n in lens]
    blocks, pages = (4096 if long_table else 512) // bs + 4, sum(need) + 1
    table, free = np.zeros((R, blocks), np.int32), list(1 + rng.permutation(pages - 1))
    for r, n in enumerate(need):
        table[r, :n] = [free.pop() for _ in range(n)]
    Q, KC, VC = up(R, nh * hd), up(pages, nkv, bs, hd), up(pages, nkv, vd, bs)
    TBL, QS, CL = rt.upload(table), rt.upload(np.arange(R + 1, dtype=np.int32)), rt.upload(np.array(lens, np.int32))
    ws = rt.zeros((k.zk_attention_bf16_workspace(R, nh, vd, 513) // 4,), "float32")
    got = []
    for once in (0, 1):
        out = rt.zeros((R, nh * vd), "bfloat16")
        k.zk_attention_bf16_once(Q.ptr, nh * hd, KC.ptr, VC.ptr, TBL.ptr, blocks, QS.ptr, CL.ptr, out.ptr, R, 0, 1, 513, nh, nkv, hd, bs, hd ** -0.5,
                                 0.0, 0, 64, ws.ptr, ws.nbytes, 0, 0, 0, 0, vd, 0, None, None, 0, 0, once, rt.stream)
        got.append(rt.download(out))
    assert np.array_equal(*got) and got[0].any(axis=1).all()
