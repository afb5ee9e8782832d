"""Products of one row that make their own norm: the bits of the norm's kernel followed by the product's, for rows by the narrow and the wide
kernel's order of sums, every kernel that takes such a row, activations and planes of partial sums."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def inputs(K, parts, seed):
    from zse_amd.runtime.device import Runtime
    from zse_amd.weights.safetensors import f32_to_bf16_bits
    rt = Runtime.get()
    k = rt.kernels("bfloat16")
    rng = np.random.default_rng(seed)
    f32 = lambda *shape: rng.standard_normal(shape, dtype=np.float32)
    bits = lambda x: rt.upload(f32_to_bf16_bits(np.ascontiguousarray(x)), "bfloat16")
    sub = rt.upload(f32(parts, K)) if parts else bits(f32(1, K))
    return rt, k, rng, f32, bits, sub, f32(1, K), rt.upload(0.3 * f32(K)), rt.upload(0.3 * f32(K))


def strips(rt, k, bits, f32, rows, K):
    W, S = bits(f32(rows, K) * np.float32(K ** -0.5)), rt.empty((-(-rows // 16) * 16, K), "bfloat16")
    k.zk_strip_layout(W.ptr, S.ptr, rows, K, rt.stream)
    return S


# K of one to sixteen waves of the wide kernel and one to seven of the narrow one's vectors; 5 to 512 strips straight from memory, 513 and 600 by
# three a block, 897 by four
@pytest.mark.parametrize("K,N", [(256, 80), (1024, 4096), (1792, 16 * 30), (2048, 8192), (2304, 16 * 513), (2304, 16 * 600), (3584, 16 * 897), (4096, 80), (3328, 16 * 520)])
@pytest.mark.parametrize("parts", [0, 1, 3, 4, 5, 6])
def test_gated(K, N, parts):
    rt, k, rng, f32, bits, sub, h, wp, wn = inputs(K, parts, K + N + parts)
    S = strips(rt, k, bits, f32, 2 * N, K)
    h0, h1, out = rt.upload(h), rt.zeros((1, K), "float32"), rt.empty((1, K), "bfloat16")
    ref, got = rt.zeros((1, N), "bfloat16"), rt.zeros((1, N), "bfloat16")
    uo = parts % 2
    k.zk_norm_gated_bf16(sub.ptr, parts, wp.ptr, 1e-6, uo, h0.ptr, h1.ptr, wn.ptr, 1e-5, uo, S.ptr, got.ptr, N, K, 2,
                         1 + 2 * uo, rt.stream)
    assert np.array_equal(rt.download(h0), h)              # the old stream is left alone
    k.zk_norm_add_norm(sub.ptr, parts, wp.ptr, 1e-6, uo, h0.ptr, wn.ptr, 1e-5, uo, out.ptr, 1, K, rt.stream)
    k.zk_gemm_bf16(out.ptr, K, S.ptr, ref.ptr, N, 0, 1, N, K, 2, 0.0, 1, None, 0, None, rt.stream)
    assert np.array_equal(rt.download(h1), rt.download(h0))
    assert np.array_equal(rt.download(ref), rt.download(got)) and rt.download(got).any()


@pytest.mark.parametrize("K,nh,nkv,hd", [(256, 4, 2, 64), (1024, 8, 2, 128), (1280, 3, 0, 32), (2304, 8, 4, 256), (4096, 32, 16, 128), (2048, 2, 1, 16)])
@pytest.mark.parametrize("parts", [0, 4, 5])
def test_rotating(K, nh, nkv, hd, parts):
    rt, k, rng, f32, bits, sub, h, wp, wn = inputs(K, parts, K + nh + parts)
    N, bs = (nh + 2 * nkv) * hd, 16
    S = strips(rt, k, bits, f32, N, K)
    pos, slot = rt.upload(np.array([4321], np.int32)), rt.upload(np.array([bs + 3], np.int32))
    freq = rt.upload((10000.0 ** (-np.arange(hd // 2) * 2 / hd)).astype(np.float32))
    h0, h1, out = rt.upload(h), rt.zeros((1, K), "float32"), rt.empty((1, K), "bfloat16")
    res = []
    for own in (1, 0):
        Q, kc, vc = rt.zeros((1, N), "bfloat16"), rt.zeros((2 * bs * max(nkv, 1) * hd,), "bfloat16"), rt.zeros((2 * bs * max(nkv, 1) * hd,), "bfloat16")
        tail = (pos.ptr, slot.ptr if nkv else None, freq.ptr, kc.ptr, vc.ptr, nh, nkv, hd, bs, 1, rt.stream)
        if own:
            k.zk_norm_qkv_rope_bf16(sub.ptr, parts, wp.ptr, 1e-6, 1, h0.ptr, h1.ptr, wn.ptr, 1e-6, 1, S.ptr, Q.ptr, N, K, 3, *tail)
            assert np.array_equal(rt.download(h0), h)
        else:
            k.zk_norm_add_norm(sub.ptr, parts, wp.ptr, 1e-6, 1, h0.ptr, wn.ptr, 1e-6, 1, out.ptr, 1, K, rt.stream)
            k.zk_qkv_rope_bf16(out.ptr, K, S.ptr, Q.ptr, N, 1, K, 1, *tail)
        res.append([rt.download(t) for t in (Q, kc, vc)])
    assert np.array_equal(rt.download(h1), rt.download(h0))
    assert all(np.array_equal(a, b) for a, b in zip(*res)) and res[0][0].any()


def test_refused():
    rt, k, rng, f32, bits, sub, h, wp, wn = inputs(256, 0, 1)
    S, C, h0, h1 = strips(rt, k, bits, f32, 160, 256), rt.zeros((1, 80), "bfloat16"), rt.upload(h), rt.zeros((1, 256), "float32")
    good = [sub.ptr, 0, wp.ptr, 1e-6, 1, h0.ptr, h1.ptr, wn.ptr, 1e-6, 1, S.ptr, C.ptr, 80, 256, 2, 1, rt.stream]
    for place, value in ((6, h0.ptr), (13, 320), (13, 8192), (12, 72), (14, 0), (14, 6), (15, 0), (0, sub.ptr + 2), (1, 7), (2, None)):
        bad = list(good)
        bad[place] = value
        with pytest.raises(Exception):
            k.zk_norm_gated_bf16(*bad)
