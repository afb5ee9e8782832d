"""Decoded tokens' attention on 16-wide tiles at the edges of its waves (32 or 64 keys) and blocks (128; 256 behind wide tables), against 64-bit arithmetic."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# pages of four keys (values in two pieces) and more; sixteen heads over one with values of 256 channels (the most LDS);
# values half and twice as wide as keys; a window with first keys kept, shorter than the context
@pytest.mark.parametrize("nh,nkv,hd,vd,bs,window,keep", [(4, 2, 32, 32, 4, 0, 0), (16, 1, 256, 256, 16, 0, 0), (8, 4, 256, 128, 8, 0, 0),
                                                         (6, 2, 64, 128, 64, 130, 0), (2, 1, 128, 128, 4, 97, 5), (16, 1, 128, 256, 4, 300, 3)])
@pytest.mark.parametrize("long_table", [False, True])
def test_edges(nh, nkv, hd, vd, bs, window, keep, long_table):
    from zse_amd.runtime.device import Runtime
    from zse_amd.weights.safetensors import bf16_bits_to_f32, f32_to_bf16_bits
    rt = Runtime.get()
    k = rt.kernels("bfloat16")
    rng = np.random.default_rng(nh + hd + bs)
    draw = lambda *shape: bf16_bits_to_f32(f32_to_bf16_bits(rng.normal(size=shape).astype(np.float32)))
    up = lambda x: rt.upload(f32_to_bf16_bits(np.ascontiguousarray(x, np.float32)), "bfloat16")
    lens = [1, 31, 32, 33, 127, 128, 129, 255, 257, 700]
    R, blocks = len(lens), (5000 if long_table else 700) // bs + 2
    pages = sum(-(-n // bs) for n in lens) + 1
    kc, vc = np.zeros((pages, nkv, bs, hd), np.float32), np.zeros((pages, nkv, vd, bs), np.float32)
    table, free = np.full((R, blocks), -1, np.int32), list(1 + rng.permutation(pages - 1))
    q, want = draw(R, nh, hd), np.zeros((R, nh, vd))
    for r, n in enumerate(lens):
        ks, vs = draw(n, nkv, hd), draw(n, nkv, vd)
        sees = [j for j in range(n) if not window or j > n - 1 - window or j < keep]
        for j in range(n):
            if j % bs == 0 and (not window or j + bs > n - window or j < keep):      # pages out of sight are given back
                table[r, j // bs] = free.pop()
            page = table[r, j // bs]
            if page >= 0:
                kc[page, :, j % bs], vc[page, :, :, j % bs] = ks[j], vs[j]
        for h in range(nh):
            g = h // (nh // nkv)
            s = 20 * np.tanh(ks[sees, g].astype(np.float64) @ q[r, h] * hd ** -0.5 / 20)
            w = np.exp(s - s.max())
            want[r, h] = w @ vs[sees, g].astype(np.float64) / w.sum()
    Q, KC, VC, TBL = up(q), up(kc), up(vc), rt.upload(table)
    QS, CL = rt.upload(np.arange(R + 1, dtype=np.int32)), rt.upload(np.array(lens, np.int32))
    ws = rt.zeros((k.zk_attention_bf16_workspace(R, nh, vd, 900) // 4,), "float32")
    got = []
    for chunk in (32, 64):
        out = rt.zeros((R, nh, vd), "bfloat16")
        k.zk_attention_bf16_sized(Q.ptr, nh * hd, KC.ptr, VC.ptr, TBL.ptr, blocks, QS.ptr, CL.ptr, out.ptr, R, 0, 1, 900, nh, nkv, hd, bs,
                                  hd ** -0.5, 20.0, window, chunk, ws.ptr, ws.nbytes, 0, 0, 0, 0, vd, keep, rt.stream)
        got.append(rt.download_f32(out).reshape(R, nh, vd))
    # a weight rounded to 8 bits of mantissa in front of a value (2^-9 of it), the result rounded likewise, values of up to 5
    assert max(np.abs(x - want).max() for x in got) < 2 * 2.0 ** -9 * 5
    if not long_table:          # there the number asked for does not say where the keys are cut
        assert np.array_equal(got[0], got[1])
