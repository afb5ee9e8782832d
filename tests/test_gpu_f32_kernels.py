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
# eight waves' steps of 32, odd and with rows further apart than K (in tiles of 16 and 32; of 64 below)
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


# Tiles of 64 x 64 (1,024 of them or more) with ragged last ones, and of the other sizes; K of fewer values than a
# load takes, of one and two steps (one and two waves), around the steps of eight waves and odd; rows and
# weights that begin at any float's address
@pytest.mark.parametrize("M,N", [(129, 22000), (40, 70001), (17, 300), (16, 17000), (2, 50)])
@pytest.mark.parametrize("K,gap,shift", [(1, 0, 0), (3, 1, 1), (4, 0, 0), (5, 0, 3), (31, 0, 0), (32, 4, 0), (36, 0, 1), (63, 1, 0), (64, 0, 2),
                                         (65, 0, 0), (260, 4, 0), (544, 0, 1), (801, 2, 0)])
def test_product_tiles_and_addresses(rt, M, N, K, gap, shift):
    k = rt.kernels("float32")
    rng = np.random.default_rng(M + K)
    a, w = rng.normal(size=(M, K + gap)).astype(np.float32), rng.normal(size=(N, K)).astype(np.float32)
    a[:, K:] = np.nan                                       # nothing between the rows is used
    pad = lambda x: np.concatenate([np.full(shift, np.nan, np.float32), x.ravel(), np.full(4, np.nan, np.float32)])
    A, W = rt.upload(pad(a)), rt.upload(pad(w))
    C, one = rt.upload(np.full((M, N + 3), 7.0, np.float32)), rt.empty((1, N), "float32")
    k.zk_gemm_plain(A.ptr + 4 * shift, K + gap, W.ptr + 4 * shift, C.ptr, N + 3, 1, M, N, K, rt.stream)
    got = rt.download(C)
    want = a[:, :K].astype(np.float64) @ w.astype(np.float64).T
    assert np.abs(got[:, :N] - want).max() < 8 * 2.0 ** -24 * max(K, 8)        # as above
    assert (got[:, N:] == 7.0).all()
    for m in {0, M // 2, M - 1}:
        k.zk_gemm_plain(A.ptr + 4 * (shift + m * (K + gap)), K + gap, W.ptr + 4 * shift, one.ptr, N, 1, 1, N, K, rt.stream)
        assert np.array_equal(rt.download(one)[0], got[m, :N]), m


# More than sixteen rows, K of 512 or more: sizes at which each of the tiles from 16 x 16 to 64 x 64 has the least price,
# with ragged last rows and columns, K a whole number of steps, of fours, and odd
@pytest.mark.parametrize("M,N,K", [(21, 102, 516), (22, 132, 513), (19, 2057, 516), (17, 2087, 513), (17, 4548, 516), (17, 4269, 513),
                                   (33, 4419, 512), (33, 4185, 513), (17, 8279, 512), (17, 8988, 515), (33, 8266, 512), (33, 8332, 513),
                                   (97, 6165, 516), (98, 6300, 513), (303, 1024, 4096)])
def test_product_tiles_by_price(rt, M, N, K):
    test_product(rt, M, N, K, 0)


# heads, key heads (one to seventeen heads a key head), sizes of keys and values, page, window, first keys kept
@pytest.mark.parametrize("nh,nkv,hd,vd,bs,window,keep", [(4, 2, 64, 64, 16, 0, 0), (3, 1, 20, 36, 4, 7, 0), (17, 1, 128, 128, 16, 70, 3),
                                                         (6, 6, 256, 256, 8, 0, 0), (10, 2, 132, 64, 32, 33, 0), (16, 1, 4, 4, 1, 0, 0)])
def test_attention(rt, nh, nkv, hd, vd, bs, window, keep):
    k = rt.kernels("float32")
    rng = np.random.default_rng(nh * hd + bs)
    reqs = [(60, 9), (0, 5), (200, 1), (63, 2), (1, 1)]            # tokens before, tokens: runs that share blocks
    pages = sum(-(-(a + n) // bs) for a, n in reqs) + 1
    kc, vc = (np.full((pages, nkv, bs, d), np.nan, np.float32) for d in (hd, vd))
    table = np.full((len(reqs), max(-(-(a + n) // bs) for a, n in reqs)), -1, np.int32)
    q, pos, own, want, seen_by = [], [], [], [], []
    sinks, free = rng.normal(size=nh).astype(np.float32), list(rng.permutation(pages))
    gates = rng.normal(size=(sum(n for _, n in reqs) + 1, nh)).astype(np.float32)
    for r, (past, n) in enumerate(reqs):
        ks, vs, qs = (rng.normal(size=(m, g, d)).astype(np.float32) for m, g, d in ((past + n, nkv, hd), (past + n, nkv, vd), (n, nh, hd)))
        if r == 0:
            vs[past + n - 1] = np.inf               # the last token's own value: no earlier token of its block sees it
        for j in range(past + n):
            if j % bs == 0:
                table[r, j // bs] = free.pop()
            kc[table[r, j // bs], :, j % bs], vc[table[r, j // bs], :, j % bs] = ks[j], vs[j]
        for i in range(n):
            p = past + i
            sees = [j for j in range(p + 1) if not window or j > p - window or j < keep]
            o = np.zeros((nh, vd))
            for h in range(nh):
                g = h // (nh // nkv)
                s = 30 * np.tanh(ks[sees, g].astype(np.float64) @ qs[i, h].astype(np.float64) * 0.2 / 30)
                w = np.exp(s - s.max())
                with np.errstate(all="ignore"):
                    o[h] = w @ vs[sees, g].astype(np.float64) / (w.sum() + np.exp(sinks[h] - s.max())) / (1 + np.exp(-gates[len(q), h]))
            q.append(qs[i]), pos.append(p), own.append(r), want.append(o)
        if r == 1:                                  # a padding row between two requests
            q.append(np.zeros((nh, hd), np.float32)), pos.append(-1), own.append(0), want.append(np.zeros((nh, vd)))
    T = len(q)
    Q, KC, VC, TBL, G, S = (rt.upload(np.ascontiguousarray(x)) for x in (np.stack(q), kc, vc, table, gates, sinks))
    POS, REQ, OUT = rt.upload(np.array(pos, np.int32)), rt.upload(np.array(own, np.int32)), rt.zeros((T, nh, vd), "float32")

    def run(t, n):
        k.zk_attention_plain_gated(Q.ptr + 4 * t * nh * hd, nh * hd, KC.ptr, VC.ptr, TBL.ptr, table.shape[1], REQ.ptr + 4 * t,
                                   POS.ptr + 4 * t, OUT.ptr + 4 * t * nh * vd, n, nh, nkv, hd, vd, bs, 0.2, 30.0, window, 0, None, 0, S.ptr,
                                   0, 0, 0, keep, G.ptr + 4 * t * nh, nh, rt.stream)
        return rt.download(OUT)
    got, want = run(0, T), np.stack(want)
    fine = np.isfinite(want)
    assert np.array_equal(fine, np.isfinite(got)) and not fine[8].all() and fine[:8].all()
    # scores of up to about hd sums, weights by exp of them: hd + 200 roundings of 2^-24, eight times over
    assert np.abs(got[fine] - want[fine]).max() < 8 * 2.0 ** -24 * (hd + 200)
    rt.zero_(OUT)
    for t in range(T):                              # each token alone: the same bits
        alone = run(t, 1)
    assert np.array_equal(alone[9:], got[9:]) and np.array_equal(alone[:8], got[:8])


# Key heads of 65 to 128 channels, whose keys and values are asked for a piece of 16 ahead: ragged and full sizes of both,
# pieces at both ends of a tile that no row sees, pages of fewer keys than a piece
@pytest.mark.parametrize("nh,nkv,hd,vd,bs,window,keep", [(4, 2, 68, 4, 16, 0, 0), (8, 2, 128, 128, 16, 0, 0), (8, 8, 100, 64, 4, 20, 0),
                                                         (2, 1, 128, 4, 16, 33, 17), (5, 1, 96, 100, 8, 0, 0)])
def test_attention_a_piece_ahead(rt, nh, nkv, hd, vd, bs, window, keep):
    test_attention(rt, nh, nkv, hd, vd, bs, window, keep)


# One request whose tokens share a block.  A value that is not finite lies in a piece of 16 keys of which
# every row sees several more: at the last token's own place (hidden from the tokens before it), or at a place
# that a window shows to the first tokens only.
@pytest.mark.parametrize("nh,nkv,past,n,window,at", [(1, 1, 70, 9, 0, 78), (4, 2, 72, 8, 0, 79), (2, 2, 70, 9, 8, 66),
                                                     (16, 1, 140, 1, 0, 3), (3, 1, 125, 5, 0, 127)])
@pytest.mark.parametrize("what", [np.inf, -np.inf, np.nan])
def test_a_value_changes_only_the_rows_that_see_it(rt, nh, nkv, past, n, window, at, what):
    k = rt.kernels("float32")
    rng = np.random.default_rng(past + at)
    hd, vd, bs, ctx = 64, 128, 16, past + n
    pages = -(-ctx // bs)
    kc, vc = (rng.normal(size=(pages, nkv, bs, d)).astype(np.float32) for d in (hd, vd))
    q = rng.normal(size=(n, nh, hd)).astype(np.float32)
    bad = vc.copy()
    bad[at // bs, :, at % bs, ::3] = what
    Q, KC, TBL = rt.upload(q), rt.upload(kc), rt.upload(np.arange(pages, dtype=np.int32)[None])
    POS, REQ, OUT = rt.upload(np.arange(past, ctx, dtype=np.int32)), rt.upload(np.zeros(n, np.int32)), rt.zeros((n, nh, vd), "float32")

    def run(v, t, m):
        V = rt.upload(v)
        k.zk_attention_plain_gated(Q.ptr + 4 * t * nh * hd, nh * hd, KC.ptr, V.ptr, TBL.ptr, pages, REQ.ptr + 4 * t, POS.ptr + 4 * t,
                                   OUT.ptr + 4 * t * nh * vd, m, nh, nkv, hd, vd, bs, 0.2, 0.0, window, 0, None, 0, None, 0, 0, 0, 0,
                                   None, 0, rt.stream)
        return rt.download(OUT)
    fine, got = run(vc, 0, n), run(bad, 0, n)
    for i in range(n):
        sees = at <= past + i and not (window and at <= past + i - window)
        clean = np.ones(vd, bool)
        clean[::3] = not sees
        assert np.array_equal(got[i][:, clean], fine[i][:, clean]), i       # the others' bits stay
        assert np.isfinite(got[i][:, clean]).all() and not np.isfinite(got[i][:, ~clean]).any(), i
    for t in range(n):                              # and each token alone has the bits that it has in company
        alone = run(bad, t, 1)
    assert np.array_equal(alone, got, equal_nan=True)


def test_rows_of_the_cache_past_2_to_the_31(rt):
    # the cache's row of a key (page, key head, place) has more than 31 bits; one page of it is filled and read
    k = rt.kernels("float32")
    nh, d, bs, page, n = 3, 4, 16, 1 << 27, 13
    rng = np.random.default_rng(0)
    kv = rng.normal(size=(bs, d)).astype(np.float32)
    cache, small = rt.empty((page + 1, 1, bs, d), "float32"), rt.upload(kv)
    rt.copy_h2d(cache.ptr + 4 * page * bs * d, kv)
    Q, O = rt.upload(rng.normal(size=(n, nh, d)).astype(np.float32)), rt.empty((n, nh, d), "float32")
    REQ, POS = rt.upload(np.zeros(n, np.int32)), rt.upload(np.arange(n, dtype=np.int32))

    def run(c, at):
        TBL = rt.upload(np.array([[at]], np.int32))
        k.zk_attention_plain(Q.ptr, nh * d, c.ptr, c.ptr, TBL.ptr, 1, REQ.ptr, POS.ptr, O.ptr, n, nh, 1, d, bs, 0.5, 0.0, 0, 0, rt.stream)
        return rt.download(O)
    assert np.array_equal(run(cache, page), run(small, 0))


def test_more_tokens_than_one_launch_holds(rt):
    # sixteen heads over one: a block a token, of 512 threads
    k = rt.kernels("float32")
    T, nh, d, bs = (1 << 23) + 1000, 16, 4, 8
    rng = np.random.default_rng(0)
    kc, vc = (rt.upload(rng.normal(size=(1, 1, bs, d)).astype(np.float32)) for _ in range(2))
    TBL, REQ, POS = rt.upload(np.zeros((1, 1), np.int32)), rt.upload(np.zeros(T, np.int32)), rt.upload(np.arange(T, dtype=np.int32) % bs)
    Q, O, few = rt.empty((T, nh, d), "float32"), rt.empty((T, nh, d), "float32"), rt.empty((512, nh, d), "float32")
    k.zk_fill_normal(Q.ptr, 0, Q.numel, 5, 1, 0.0, 1.0, rt.stream)

    def run(t, n, out):
        k.zk_attention_plain(Q.ptr + 4 * t * nh * d, nh * d, kc.ptr, vc.ptr, TBL.ptr, 1, REQ.ptr + 4 * t, POS.ptr + 4 * t, out, n, nh, 1, d, bs,
                             0.5, 0.0, 0, 0, rt.stream)
    run(0, T, O.ptr)
    for t in (0, (1 << 22) - 256, (1 << 23) - 256, T - 512):
        run(t, 512, few.ptr)
        assert np.array_equal(rt.download(O.rows(t, t + 512)), rt.download(few)), t


def test_more_blocks_of_columns_than_one_launch_holds(rt):
    # a launch holds less than 2^32 threads: 2^28 columns and more leave in several
    k = rt.kernels("float32")
    M, N, K = 2, (1 << 28) + 2000, 4
    W, C = rt.empty((N, K), "float32"), rt.empty((M, N), "float32")
    k.zk_fill_normal(W.ptr, 0, W.numel, 5, 1, 0.0, 1.0, rt.stream)
    a = np.random.default_rng(0).normal(size=(M, K)).astype(np.float32)
    A = rt.upload(a)
    k.zk_gemm_plain(A.ptr, K, W.ptr, C.ptr, N, 1, M, N, K, rt.stream)
    few = rt.empty((M, 2048), "float32")
    for n0 in (0, (1 << 27) - 1024, (1 << 28) - 1024, N - 2048):
        k.zk_gemm_plain(A.ptr, K, W.ptr + 4 * K * n0, few.ptr, 2048, 1, M, 2048, K, rt.stream)
        want = rt.download(few)
        for m in range(M):
            assert np.array_equal(rt.download(type(C)(C.ptr + 4 * (m * N + n0), (2048,), "float32")), want[m]), (n0, m)


# Many short runs: blocks that take eight (four) runs at once, one with all its waves, and several rounds of runs, with
# padding rows between; the same tokens a few at a time go a run a block
@pytest.mark.parametrize("nh,nkv,hd,vd,window,keep,chunk,turned", [(8, 8, 64, 64, 0, 0, 0, 0), (9, 3, 20, 128, 70, 3, 0, 0), (16, 8, 128, 128, 0, 0, 96, 1),
                                                                   (6, 6, 256, 64, 40, 0, 0, 0), (34, 17, 4, 8, 0, 0, 0, 1)])
def test_many_short_runs(rt, nh, nkv, hd, vd, window, keep, chunk, turned):
    k = rt.kernels("float32")
    rng = np.random.default_rng(nh + hd)
    bs, slots, own, pos = 16, 24, [], []
    lens = [rng.integers(1, 64), 64, 65, 128, 129, 250, 300, 600]            # keys a run may reach, by regions of the step
    while len(own) < 3000:
        top, n = int(lens[len(own) * len(lens) // 3001]), int(rng.choice([1, 1, 2, 3, 5, 9, 20]))
        first = int(rng.integers(0, max(top - n, 0) + 1))
        own += [len(own) % slots] * n
        pos += list(range(first, first + n))
        if rng.random() < 0.1:
            own.append(0), pos.append(-1)
    T, per = len(own), 640 // bs
    Q, KC, VC = (rt.upload(rng.normal(size=s).astype(np.float32)) for s in ((T, nh, hd), (slots * per, nkv, bs, hd), (slots * per, nkv, bs, vd)))
    TBL, S = rt.upload(rng.permutation(slots * per).astype(np.int32).reshape(slots, per)), rt.upload(rng.normal(size=nh).astype(np.float32))
    POS, REQ, F = rt.upload(np.array(pos, np.int32)), rt.upload(np.array(own, np.int32)), rt.upload(rng.random(vd // 2).astype(np.float32))
    OUT = rt.upload(np.full((T, nh, vd), 7.0, np.float32))

    def run(t, n):
        k.zk_attention_plain_gated(Q.ptr + 4 * t * nh * hd, nh * hd, KC.ptr, VC.ptr, TBL.ptr, per, REQ.ptr + 4 * t, POS.ptr + 4 * t,
                                   OUT.ptr + 4 * t * nh * vd, n, nh, nkv, hd, vd, bs, 0.2, 0.0, window, 0, F.ptr if turned else None, 0, S.ptr,
                                   0, chunk, 0, keep, None, 0, rt.stream)
    run(0, T)
    together = rt.download(OUT)
    rt.zero_(OUT)
    for t in range(0, T, 61):
        run(t, min(61, T - t))
    alone = rt.download(OUT)
    assert np.isfinite(together).all() and np.array_equal(together, alone)
    assert (together[np.array(pos) < 0] == 0).all() and (np.abs(together[np.array(pos) >= 0]).max(axis=(1, 2)) > 0).all()
