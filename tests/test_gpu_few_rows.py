"""Products of up to 16 rows whose addresses go by whole groups of steps, or K in ranges over few long strips, and decoded
tokens' attention in its forms for few and for many blocks: against 64-bit arithmetic, and the same bits where the sums are the same."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def dev():
    from zse_amd.runtime.device import Runtime
    rt = Runtime.get()
    return rt, rt.kernels("bfloat16")


# one group; not whole (288); a last strip that is not full; few long strips in ranges (two, four, five of them), few short ones
# and 224 that nearly fill the chip (no ranges); more strips than compute units in ranges
@pytest.mark.parametrize("N,K,ranges", [(48, 256, 0), (64, 288, 0), (1000, 1024, 0), (2048, 8192, 2), (1024, 4096, 4), (2304, 9216, 5),
                                        (2048, 2048, 0), (3584, 4096, 0), (4608, 4096, 4)])
@pytest.mark.parametrize("gated", [0, 1])
def test_products(N, K, ranges, gated):
    from zse_amd.weights.safetensors import bf16_bits_to_f32, f32_to_bf16_bits
    rt, k = dev()
    if gated and N * K > 1 << 22 or gated and N % 16:
        pytest.skip("the gated product has no ranges and takes whole strips")
    rng = np.random.default_rng(N + K)
    bits = lambda *shape: f32_to_bf16_bits(rng.normal(size=shape).astype(np.float32) * K ** -0.25)
    a, w = bits(16, K), bits(N * (1 + gated), K)
    A, W = rt.upload(a, "bfloat16"), rt.upload(w, "bfloat16")
    S = rt.empty((-(-w.shape[0] // 16) * 16, K), "bfloat16")
    k.zk_strip_layout(W.ptr, S.ptr, *w.shape, rt.stream)
    ws = rt.zeros((k.zk_gemm_bf16_workspace() // 4,), "float32")
    want = bf16_bits_to_f32(a).astype(np.float64) @ bf16_bits_to_f32(w).astype(np.float64).T
    if gated:
        want = np.maximum(want[:, :N], 0) * want[:, N:]
    rows = {}
    for M in (1, 7, 16):
        for ldc in (N, N + 8):
            C = rt.upload(np.full((M + 1, ldc), 0x4040, np.uint16), "bfloat16")
            k.zk_gemm_bf16(A.ptr, K, S.ptr, C.ptr, ldc, 0, M, N, K, 5 if gated else 0, 0.0, 1, ws.ptr, ws.nbytes, None, rt.stream)
            got = rt.download_f32(C)
            # a result rounded to 8 bits of mantissa; K float additions of products of size K^-0.5
            assert (np.abs(got[:M, :N] - want[:M]) <= np.abs(want[:M]) * 2.0 ** -8 + 1e-4 * (1 + 3 * gated)).all(), (M, ldc)
            assert (got[M:] == 3.0).all() and (got[:, N:] == 3.0).all()
            rows.setdefault("whole", got[0, :N])
            assert np.array_equal(got[0, :N], rows["whole"])       # a row does not know of the others
        if gated:
            continue
        parts = ctypes.c_int(0)
        C = rt.zeros((M, N), "bfloat16")
        k.zk_gemm_bf16(A.ptr, K, S.ptr, C.ptr, N, 0, M, N, K, 0, 0.0, 1, ws.ptr, ws.nbytes, ctypes.byref(parts), rt.stream)
        assert parts.value == ranges, (M, parts.value)
        if ranges:
            planes = rt.download(ws)[:ranges * M * N].reshape(ranges, M, N)
            # float sums of K products of size K^-0.5, in another order
            assert np.abs(planes.astype(np.float64).sum(0) - want[:M]).max() < 2e-5 * max(1.0, np.abs(want).max())
            rows.setdefault("ranges", planes[:, 0])
            assert np.array_equal(planes[:, 0], rows["ranges"])


@pytest.mark.parametrize("nh,nkv,hd,K", [(4, 2, 64, 256), (2, 1, 256, 2304), (3, 1, 16, 512), (4, 0, 128, 1024)])
@pytest.mark.parametrize("M", [1, 16])
def test_the_rotating_product_gives_the_bits_of_product_and_rotation(M, nh, nkv, hd, K):
    from zse_amd.weights.safetensors import f32_to_bf16_bits
    rt, k = dev()
    rng = np.random.default_rng(hd + K)
    N, bs = (nh + 2 * nkv) * hd, 16
    up = lambda x: rt.upload(f32_to_bf16_bits(np.ascontiguousarray(x, np.float32)), "bfloat16")
    A, W, S = up(rng.normal(size=(M, K))), up(rng.normal(size=(N, K)) * K ** -0.5), rt.empty((N, K), "bfloat16")
    k.zk_strip_layout(W.ptr, S.ptr, N, K, rt.stream)
    pos = rt.upload(rng.integers(0, 8000, M).astype(np.int32))
    slots = rt.upload((rng.permutation(2 * bs)[:M]).astype(np.int32))
    freq = rt.upload((10000.0 ** (-np.arange(hd // 2) * 2 / hd)).astype(np.float32))
    got = []
    for fused in (True, False):
        Q = rt.zeros((M, N), "bfloat16")
        kc, vc = rt.zeros((2 * max(nkv, 1) * bs * hd,), "bfloat16"), rt.zeros((2 * max(nkv, 1) * bs * hd,), "bfloat16")
        if fused:
            k.zk_qkv_rope_bf16(A.ptr, K, S.ptr, Q.ptr, N, M, K, 1, pos.ptr, slots.ptr if nkv else None, freq.ptr, kc.ptr, vc.ptr, nh, nkv,
                               hd, bs, 1, rt.stream)
        else:
            k.zk_gemm_bf16(A.ptr, K, S.ptr, Q.ptr, N, 0, M, N, K, 0, 0.0, 1, None, 0, None, rt.stream)
            k.zk_rope_cache_write(Q.ptr, pos.ptr, slots.ptr if nkv else None, freq.ptr, hd, kc.ptr, vc.ptr, M, nh, nkv, hd, bs, 1, rt.stream)
        got.append((rt.download_f32(Q)[:, :nh * hd], rt.download_f32(kc), rt.download_f32(vc)))
    for a, b in zip(*got):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("nh,nkv,hd", [(8, 4, 256), (8, 2, 128), (16, 1, 64)])
def test_attention_of_few_and_many_blocks_and_with_a_window_that_shows_all(nh, nkv, hd):
    """Requests of one to 78 parts of 128 keys (32 of which the join asks for at once, and those up to 64 eight at a time): alone,
    among so many that the chip is full, and behind a window as long as the longest context, whose parts are counted from the request's
    length: the same bits, those of 64-bit sums but for the rounding of weights and results."""
    from test_gpu_stream_attention import plain, rounded
    from zse_amd.weights.safetensors import f32_to_bf16_bits
    rt, k = dev()
    rng = np.random.default_rng(hd)
    up = lambda x: rt.upload(f32_to_bf16_bits(np.ascontiguousarray(x, np.float32)), "bfloat16")
    bs, lens = 16, [1, 128, 129, 1000, 1030, 2049, 4100, 9900, 5200, 8192]
    ends = np.cumsum([0] + [-(-n // bs) for n in lens])
    keys, values = rng.normal(size=(ends[-1], nkv, bs, hd)), rng.normal(size=(ends[-1], nkv, hd, bs))
    kc, vc = up(keys), up(values)
    q = rng.normal(size=(len(lens), nh, hd)).astype(np.float32)

    def run(copies, window, chunk):
        R = len(lens) * copies
        blocks = 9984 // bs          # (decode_chunk 32: parts of 128 keys beside any table)
        table = np.full((R, blocks), -1, np.int32)
        for r in range(R):
            a, b = ends[r % len(lens)], ends[r % len(lens) + 1]
            table[r, :b - a] = np.arange(a, b)
        Q, TBL = up(np.tile(q, (copies, 1, 1))), rt.upload(table)
        QS, CL = rt.upload(np.arange(R + 1, dtype=np.int32)), rt.upload(np.tile(np.array(lens, np.int32), copies))
        ws = rt.zeros((k.zk_attention_bf16_workspace(R, nh, hd, 9984) // 4,), "float32")
        out = rt.zeros((R, nh, hd), "bfloat16")
        k.zk_attention_bf16(Q.ptr, nh * hd, kc.ptr, vc.ptr, TBL.ptr, blocks, QS.ptr, CL.ptr, out.ptr, R, 0, 1, 9984, nh, nkv, hd, bs,
                            hd ** -0.5, 50.0, window, chunk, ws.ptr, ws.nbytes, rt.stream)
        return rt.download_f32(out).reshape(copies, len(lens), nh * hd)
    want = run(1, 0, 32)[0]
    assert np.isfinite(want).all() and want.any(axis=1).all()
    for i, n in enumerate(lens):
        kk = rounded(keys[ends[i]:ends[i + 1]]).transpose(0, 2, 1, 3).reshape(-1, nkv, hd)[:n].astype(np.float64)
        vv = rounded(values[ends[i]:ends[i + 1]]).transpose(0, 3, 1, 2).reshape(-1, nkv, hd)[:n].astype(np.float64)
        o, size = (plain(rounded(q[i:i + 1]).astype(np.float64), kk, v, n - 1, hd ** -0.5, 50.0, 0, 0) for v in (vv, np.abs(vv)))
        # weights rounded to 8 bits of mantissa (not in their sum), and the result's own rounding
        assert (np.abs(want[i].reshape(o.shape) - o) <= 2.0 ** -8 * (size + np.abs(o))).all(), n
    for copies, window in ((1, 9983), (12, 0), (12, 9900)):
        got = run(copies, window, 32)
        assert all(np.array_equal(x, want) for x in got), (copies, window)


# a block a token, from 2,048 of them on with the values asked for when they are stored; values in rows
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("T,nh,nkv,hd,bs,vt", [(300, 8, 4, 256, 16, 1), (2049, 8, 4, 256, 16, 1), (2047, 8, 4, 128, 4, 1), (4103, 6, 1, 32, 8, 1),
                                               (2100, 2, 1, 128, 16, 0)])
def test_rotation_and_store_of_many_tokens(dtype, T, nh, nkv, hd, bs, vt):
    from test_gpu_kernels import test_rope_and_cache_write
    assert dev()[1]._dll.zk_rope_by_token(T, nh, nkv, hd, hd, vt, 0)
    test_rope_and_cache_write(dev()[0], dtype, T, nh, nkv, hd, hd, bs, vt)


# heads, key heads, key and value channels, page, (cached, new) of each request, window, kept, cap, rising: one row; a block that is not
# full; 5, 8 and 1 tokens a block; 32 keys and one more, a tile for each wave and one more; windows that begin inside a tile, with kept
# keys; values of another width; maxima that rise
SHORT = [(8, 4, 256, 256, 16, [(0, 2)], 0, 0, 50.0, False), (6, 2, 128, 128, 16, [(0, 33), (31, 5), (100, 29)], 0, 0, 0.0, False),
         (16, 1, 256, 256, 32, [(60, 69)], 0, 0, 30.0, False), (8, 4, 256, 256, 64, [(3, 126), (0, 128)], 0, 0, 50.0, False),
         (8, 2, 128, 128, 16, [(300, 150)], 97, 0, 0.0, False), (8, 4, 256, 256, 16, [(200, 40)], 50, 37, 50.0, False),
         (4, 2, 256, 128, 16, [(10, 31)], 0, 0, 0.0, False), (4, 2, 128, 256, 16, [(0, 129)], 0, 0, 0.0, False),
         (8, 8, 128, 128, 16, [(0, 290)], 0, 0, 0.0, True)]


@pytest.mark.parametrize("case", SHORT)
def test_portions_of_few_rows(case):
    from test_gpu_stream_attention import test_portions
    from test_portion_forms import form_of
    H, G, D, E, bs, reqs, window, keep, cap, rising = case
    assert form_of(1 << 28, len(reqs), max(b for _, b in reqs), max(a + b for a, b in reqs), H, G, D, E, bs, window, 0, keep)[2] == 2
    test_portions(dev()[0], case, 0)


@pytest.mark.parametrize("H,G,D,window", [(8, 4, 256, 0), (8, 2, 128, 40)])
def test_nothing_outside_a_portions_keys_is_used(H, G, D, window):
    """Keys and values behind the last key of a page, and in pages behind the last or in front of the window, are not numbers."""
    from test_gpu_stream_attention import plain, rounded, up
    rt, k = dev()
    rng = np.random.default_rng(D)
    bs, before, n = 16, 70, 23
    ctx, blocks = before + n, 9
    kc, vc = np.full((blocks + 1, G, bs, D), np.nan, np.float32), np.full((blocks + 1, G, D, bs), np.nan, np.float32)
    q, kk, vv = (rounded(rng.normal(size=(m, h, D))) for m, h in ((n, H), (ctx, G), (ctx, G)))
    first = max(0, before - window + 1) if window else 0
    for p in range(first, ctx):
        kc[1 + p // bs, :, p % bs], vc[1 + p // bs, :, :, p % bs] = kk[p], vv[p]
    table = (1 + np.arange(blocks, dtype=np.int32)).reshape(1, -1)          # entries behind the last page lead to pages too
    out = rt.zeros((n, H * D), "bfloat16")
    ws = rt.zeros((1 << 20,), "float32")
    args = [up(rt, q.reshape(n, -1)), up(rt, kc), up(rt, vc), rt.upload(table, "int32"), rt.upload(np.array([0, n], np.int32), "int32"),
            rt.upload(np.array([ctx], np.int32), "int32")]
    k.zk_attention_bf16(args[0].ptr, H * D, args[1].ptr, args[2].ptr, args[3].ptr, blocks, args[4].ptr, args[5].ptr, out.ptr, 1, 1, n, ctx, H,
                        G, D, bs, D ** -0.5, 0.0, window, 0, ws.ptr, ws.nbytes, rt.stream)
    got = rt.download_f32(out).reshape(n, H, D)
    want = plain(q.astype(np.float64), kk.astype(np.float64), vv.astype(np.float64), before, D ** -0.5, 0.0, window, 0)
    assert np.abs(got - want).max() < 0.03
