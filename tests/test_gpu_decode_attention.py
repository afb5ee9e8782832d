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


# chunks instead of a window with a unit sink; learned sinks and gates, kept first keys; weights with 16 bits of mantissa;
# two and four key heads on one value head; values of another width; sixteen heads over one; 32-wide tiles (more heads than 16)
@pytest.mark.parametrize("nh,nkv,hd,vd,bs,window,keep,mask_chunk,sink,wide,v_shift,learned", [
    (4, 2, 128, 128, 16, 0, 0, 700, 1, 0, 0, 0), (3, 3, 32, 32, 8, 0, 0, 33, 1, 1, 0, 0), (2, 2, 256, 256, 32, 0, 0, 5000, 0, 1, 0, 0),
    (8, 2, 64, 64, 16, 700, 0, 0, 0, 1, 0, 1), (4, 4, 128, 64, 16, 333, 300, 0, 0, 0, 0, 1), (4, 2, 32, 64, 4, 0, 0, 0, 0, 1, 0, 1),
    (8, 4, 64, 64, 16, 90, 0, 0, 0, 1, 1, 0), (8, 4, 128, 128, 8, 0, 0, 0, 0, 0, 2, 0), (16, 1, 128, 128, 16, 2500, 7, 0, 0, 0, 0, 1),
    (20, 1, 64, 64, 16, 0, 0, 900, 1, 0, 0, 0)])
@pytest.mark.parametrize("wide_table", [False, True])
def test_options_and_long_contexts(nh, nkv, hd, vd, bs, window, keep, mask_chunk, sink, wide, v_shift, learned, wide_table):
    """Blocks of 128 keys (narrow tables, or a decode_chunk of 32) and of 256 (wide ones), an even and an odd
    number of blocks a request, and joins of one to 67 parts: the wide table's contexts have more than 32 of either."""
    from zse_amd.runtime.device import Runtime
    from zse_amd.weights.safetensors import bf16_bits_to_f32, f32_to_bf16_bits
    rt = Runtime.get()
    k = rt.kernels("bfloat16")
    rng = np.random.default_rng(nh + hd + window + mask_chunk)
    draw = lambda *shape: bf16_bits_to_f32(f32_to_bf16_bits(rng.normal(size=shape).astype(np.float32)))
    up = lambda x: rt.upload(f32_to_bf16_bits(np.ascontiguousarray(x, np.float32)), "bfloat16")
    lens = [1, 130, 699, 701, 1025, 4097, 8500] if wide_table else [1, 33, 129, 256, 698, 1000]
    R, blocks, maps = len(lens), (8704 if wide_table else 1024) // bs, 1 << v_shift
    pages = sum(-(-n // bs) for n in lens) + 1
    kc, vc = np.zeros((pages, nkv, bs, hd), np.float32), np.zeros((pages, nkv // maps, vd, bs), np.float32)
    table, free = np.full((R, blocks), -1, np.int32), list(1 + rng.permutation(pages - 1))
    ld = nh * hd + (nh + 7) // 8 * 8
    rows, want = draw(R, ld), np.zeros((R, nh, vd))
    sinks = draw(nh) * 3
    group = nh // nkv
    for r, n in enumerate(lens):
        ks, vs = draw(n, nkv, hd), draw(n, nkv // maps, vd)
        lo = n - 1 - (n - 1) % mask_chunk if mask_chunk else max(0, n - window) if window else 0
        sees = [j for j in range(n) if j >= lo or j < keep]
        for b in range(-(-n // bs)):
            if (b + 1) * bs > lo or b * bs < keep:          # pages out of sight are given back
                table[r, b] = free.pop()
                part = slice(b * bs, min(n, (b + 1) * bs))
                kc[table[r, b], :, :part.stop - part.start] = ks[part].transpose(1, 0, 2)
                vc[table[r, b], :, :, :part.stop - part.start] = vs[part].transpose(1, 2, 0)
        q, gate = rows[r, :nh * hd].reshape(nh, hd).astype(np.float64), rows[r, nh * hd:nh * hd + nh].astype(np.float64)
        for h in range(nh):
            # the maps of a query head lie side by side: key head (value head, map)
            g = h // (group * maps) * maps + h % maps
            s = 20 * np.tanh(ks[sees, g].astype(np.float64) @ q[h] * hd ** -0.5 / 20)
            extra = 0.0 if sink else float(sinks[h]) if learned else -np.inf
            top = max(s.max(), extra)
            w = np.exp(s - top)
            want[r, h] = w @ vs[sees, g // maps].astype(np.float64) / (w.sum() + np.exp(extra - top))
            if learned:
                want[r, h] /= 1 + np.exp(-gate[h])
    Q, KC, VC, TBL, S = up(rows), up(kc), up(vc), rt.upload(table), rt.upload(sinks.astype(np.float32))
    QS, CL = rt.upload(np.arange(R + 1, dtype=np.int32)), rt.upload(np.array(lens, np.int32))
    got = []
    for chunk, max_ctx in ((64, lens[-1]), (32, lens[-1]), (64, blocks * bs), (32, blocks * bs - 20)):
        ws = rt.zeros((k.zk_attention_bf16_workspace(R, nh, vd, max_ctx) // 4,), "float32")
        out = rt.zeros((R, nh, vd), "bfloat16")
        k.zk_attention_bf16_gated(Q.ptr, ld, KC.ptr, VC.ptr, TBL.ptr, blocks, QS.ptr, CL.ptr, out.ptr, R, 0, 1, max_ctx, nh, nkv, hd, bs,
                                  hd ** -0.5, 20.0, window, chunk, ws.ptr, ws.nbytes, mask_chunk, sink, wide, v_shift, vd, keep,
                                  S.ptr if learned else None, Q.ptr + 2 * nh * hd if learned else None, ld, rt.stream)
        got.append(rt.download_f32(out).reshape(R, nh, vd))
    # as above; the result of wide weights is rounded once
    assert max(np.abs(x - want).max() for x in got) < (1 if wide else 2) * 2.0 ** -9 * 5
    # the grid, and with it the order of the blocks, changes nothing
    assert np.array_equal(got[0], got[2]) and np.array_equal(got[1], got[3])
    if wide_table and group <= 16 and mask_chunk != 33:         # (33 keys meet no cut)
        assert not np.array_equal(got[0], got[1])           # cut after 256 keys and after 128
