"""Portions of heads of 128 and 256 channels whose tiles are copied ahead, without and with ranges of keys, against a
plain implementation in 64 bits: last blocks of a few rows (waves with no rows among them), heads that do not fill
a wave's 32 rows, pages of 16 to 64 keys, windows with kept first keys, scores whose maximum rises with every
tile, and the choice by sizes."""
import numpy as np
import pytest

from test_portion_forms import form_of

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    from zse_amd.runtime.device import Runtime
    return Runtime.get()


def rounded(x):
    from zse_amd.weights.safetensors import bf16_bits_to_f32, f32_to_bf16_bits
    return bf16_bits_to_f32(f32_to_bf16_bits(np.ascontiguousarray(x, np.float32)))


def up(rt, x):
    from zse_amd.weights.safetensors import f32_to_bf16_bits
    return rt.upload(f32_to_bf16_bits(np.ascontiguousarray(x, np.float32)), "bfloat16")


def plain(q, k, v, before, scale, cap, window, keep):
    """q [n, H, D] behind ``before`` keys of k [ctx, G, D], v [ctx, G, E]."""
    n, H, _ = q.shape
    pos, key = before + np.arange(n)[:, None], np.arange(len(k))[None]
    ok = (key <= pos) & ((key > pos - window) | (key < keep) if window else True)
    out = np.zeros((n, H, v.shape[2]))
    for h in range(H):
        g = h // (H // k.shape[1])
        s = q[:, h] @ k[:, g].T * scale
        s = np.where(ok, cap * np.tanh(s / cap) if cap else s, -np.inf)
        w = np.exp(s - s.max(1, keepdims=True))
        out[:, h] = w / w.sum(1, keepdims=True) @ v[:, g]
    return out


CASES = [
    # heads, key heads, key and value channels, page, (cached, new) of each request, window, kept, cap, rising
    (8, 4, 256, 256, 16, [(0, 64), (37, 300)], 0, 0, 50.0, False),
    (2, 2, 256, 256, 16, [(0, 1500)], 0, 0, 50.0, False),                  # a last block of one wave with rows
    (6, 2, 256, 256, 32, [(5, 97), (130, 333)], 130, 0, 0.0, False),       # 30 of a wave's 32 rows
    (4, 2, 256, 256, 64, [(700, 161)], 300, 40, 20.0, False),
    (4, 4, 256, 256, 16, [(0, 260)], 0, 0, 0.0, True),
    (8, 2, 128, 128, 16, [(0, 33), (1, 31), (900, 129)], 0, 0, 0.0, False),
    (10, 2, 128, 128, 32, [(64, 200)], 90, 7, 30.0, False),
    (4, 1, 128, 128, 16, [(300, 520)], 0, 0, 0.0, True),
    (16, 1, 128, 128, 64, [(3, 70)], 1, 0, 50.0, False),
    (4, 2, 256, 128, 16, [(40, 150)], 0, 0, 50.0, False),
    (4, 2, 128, 256, 32, [(40, 150)], 77, 33, 0.0, False),
    (4, 2, 256, 128, 16, [(231, 190)], 0, 0, 50.0, False),                # uneven heads in ranges
    (4, 2, 128, 256, 32, [(700, 150)], 300, 33, 0.0, False),
]


@pytest.mark.parametrize("mode", [0, 4, 5])           # by the sizes, four groups a block, with ranges
@pytest.mark.parametrize("case", CASES)
def test_portions(rt, case, mode):
    H, G, D, E, bs, reqs, window, keep, cap, rising = case
    kern = rt.kernels("bfloat16")
    rng = np.random.default_rng(D + E + len(reqs) + window)
    R, ctx, fresh = len(reqs), [a + b for a, b in reqs], [b for _, b in reqs]
    blocks = -(-max(ctx) // bs)
    pages = 1 + R * blocks
    table = (1 + rng.permutation(R * blocks)).astype(np.int32).reshape(R, blocks)
    kc, vc = np.zeros((pages, G, bs, D), np.float32), np.zeros((pages, G, E, bs), np.float32)
    q = rounded(rng.normal(size=(sum(fresh), H, D)))
    starts = np.concatenate([[0], np.cumsum(fresh)]).astype(np.int32)
    want = []
    for r in range(R):
        kk, vv = rng.normal(size=(ctx[r], G, D)), rounded(rng.normal(size=(ctx[r], G, E)))
        mine = q[starts[r]:starts[r + 1]]
        if rising:           # the n-th key agrees with every query the better the later it comes: about 60 maxima on the way
            q[starts[r]:starts[r + 1], :, 0] = 4.0
            kk[:, :, 0] = np.linspace(-40, 40, ctx[r])[:, None] * D ** 0.5 / 4
        kk = rounded(kk)
        for p in range(ctx[r]):
            kc[table[r, p // bs], :, p % bs], vc[table[r, p // bs], :, :, p % bs] = kk[p], vv[p]
        table[r, -(-ctx[r] // bs):] = -1
        want.append(plain(mine.astype(np.float64), kk.astype(np.float64), vv.astype(np.float64), reqs[r][0], D ** -0.5, cap, window, keep))
    want = np.concatenate(want)
    out = rt.zeros((len(q), H * E), "bfloat16")
    ws = rt.zeros((int(kern.zk_attention_bf16_portion_workspace(R * (max(fresh) + 128), H, G, E)) // 4 + 64,), "float32")
    args = [up(rt, q.reshape(len(q), -1)), up(rt, kc), up(rt, vc), rt.upload(table, "int32"), rt.upload(starts, "int32"),
            rt.upload(np.array(ctx, np.int32), "int32")]
    before = kern.zk_attention_bf16_portion_kernel(mode)
    try:
        form, tiles, stream = form_of(ws.nbytes, R, max(fresh), max(ctx), H, G, D, E, bs, window, 0, keep)
        if mode:
            # the longest block's tiles: ranges of at least four, two of them or more
            reach = min(max(ctx), window + 4 * (32 // (H // G)) - 1 if window else max(ctx))
            assert stream and form == (5 if mode == 5 and reach >= 8 * 32 else 4) and (form != 5 or tiles >= 4)
        kern.zk_attention_bf16_sized(args[0].ptr, H * D, args[1].ptr, args[2].ptr, args[3].ptr, blocks, args[4].ptr, args[5].ptr,
                                     out.ptr, R, R, max(fresh), max(ctx), H, G, D, bs, D ** -0.5, cap, window, 0, ws.ptr, ws.nbytes,
                                     0, 0, 0, 0, E, keep, rt.stream)
        got = rt.download_f32(out).reshape(want.shape)
    finally:
        kern.zk_attention_bf16_portion_kernel(before)
    # weights and results rounded to 8 bits of mantissa; values of size 1, the largest about 4.5
    assert np.abs(got - want).max() < 0.03, np.unravel_index(np.abs(got - want).argmax(), got.shape)
    assert np.linalg.norm(got - want) < 4e-3 * np.linalg.norm(want)


@pytest.mark.parametrize("mode", [0, 4, 5])
def test_pages_of_4_gib(rt, mode):
    """A page's bytes and the places in it are more than 32 bits can count: the bits of a cache of small pages."""
    kern = rt.kernels("bfloat16")
    H, G, D, n, big, small = 8, 2, 256, 288, 1 << 22, 32
    rng = np.random.default_rng(4)
    q, k, v = up(rt, rng.normal(size=(n, H * D))), rng.normal(size=(G, n, D)), rng.normal(size=(G, D, n))
    starts, ctx, out = rt.upload(np.array([0, n], np.int32)), rt.upload(np.array([n], np.int32)), rt.zeros((n, H * D), "bfloat16")
    ws = rt.zeros((int(kern.zk_attention_bf16_portion_workspace(n + 128, H, G, D)) // 4 + 64,), "float32")

    def run(kc, vc, table, bs):
        table, n_pages = rt.upload(np.array([table], np.int32)), len(table)
        before = kern.zk_attention_bf16_portion_kernel(mode)
        try:
            kern.zk_attention_bf16_sized(q.ptr, H * D, kc.ptr, vc.ptr, table.ptr, n_pages, starts.ptr, ctx.ptr, out.ptr, 1, 1, n, n, H, G, D,
                                         bs, D ** -0.5, 50.0, 0, 0, ws.ptr, ws.nbytes, 0, 0, 0, 0, D, 0, rt.stream)
            return rt.download(out)
        finally:
            kern.zk_attention_bf16_portion_kernel(before)

    from zse_amd.weights.safetensors import f32_to_bf16_bits
    bits = lambda x: f32_to_bf16_bits(np.ascontiguousarray(x, np.float32))
    want = run(up(rt, k.reshape(G, n // small, small, D).swapaxes(0, 1)), up(rt, v.reshape(G, D, n // small, small).transpose(2, 0, 1, 3)),
               list(range(n // small)), small)
    kc, vc = rt.empty((2, G, big, D), "bfloat16"), rt.empty((2, G, D, big), "bfloat16")       # 16 GiB; page 1 is the request's
    for g in range(G):
        rt.copy_h2d(kc.ptr + 2 * (G + g) * big * D, bits(k[g]))
        for d in range(D):
            rt.copy_h2d(vc.ptr + 2 * ((G + g) * D + d) * big, bits(v[g, d]))
    assert np.array_equal(run(kc, vc, [1], big), want)


@pytest.mark.parametrize("mode", [0, 4, 5])
@pytest.mark.parametrize("D,E,before,n", [(256, 256, 0, 40), (128, 128, 0, 296), (256, 256, 200, 121), (128, 256, 1000, 70), (256, 128, 0, 705)])
def test_table_entries_behind_the_last_page(rt, mode, D, E, before, n):
    """The page after a request's last one is another's and holds NaN; the last tile of keys reaches into it."""
    kern = rt.kernels("bfloat16")
    H, G, bs, ctx = 4, 2, 16, before + n
    used = -(-ctx // bs)
    assert used % 2 == 1
    rng = np.random.default_rng(n)
    q, k, v = (rounded(rng.normal(size=s)) for s in ((n, H, D), (ctx, G, D), (ctx, G, E)))
    kc, vc = np.full((used + 2, bs, G, D), np.nan, np.float32), np.full((used + 2, bs, G, E), np.nan, np.float32)
    kc[:used], vc[:used] = 0, 0
    kc[:used].reshape(-1, G, D)[:ctx], vc[:used].reshape(-1, G, E)[:ctx] = k, v
    table = np.concatenate([np.arange(used + 1), np.full(7, used + 1)]).astype(np.int32)
    out = rt.zeros((n, H * E), "bfloat16")
    ws = rt.zeros((int(kern.zk_attention_bf16_portion_workspace(n + 128, H, G, E)) // 4 + 64,), "float32")
    args = [up(rt, q.reshape(n, -1)), up(rt, kc.swapaxes(1, 2)), up(rt, vc.transpose(0, 2, 3, 1)), rt.upload(table, "int32"),
            rt.upload(np.array([0, n], np.int32), "int32"), rt.upload(np.array([ctx], np.int32), "int32")]
    mode_before = kern.zk_attention_bf16_portion_kernel(mode)
    try:
        kern.zk_attention_bf16_sized(args[0].ptr, H * D, args[1].ptr, args[2].ptr, args[3].ptr, len(table), args[4].ptr, args[5].ptr, out.ptr,
                                     1, 1, n, ctx, H, G, D, bs, D ** -0.5, 0.0, 0, 0, ws.ptr, ws.nbytes, 0, 0, 0, 0, E, 0, rt.stream)
        got = rt.download_f32(out).reshape(n, H, E)
    finally:
        kern.zk_attention_bf16_portion_kernel(mode_before)
    want = plain(q.astype(np.float64), k.astype(np.float64), v.astype(np.float64), before, D ** -0.5, 0.0, 0, 0)
    assert np.isfinite(got).all()
    assert np.linalg.norm(got - want) < 4e-3 * np.linalg.norm(want)


@pytest.mark.parametrize("H,G,D,rows,ctx", [(8, 4, 256, 512, 4096), (32, 16, 128, 512, 4096)])
def test_ranges_without_room_for_them(rt, H, G, D, rows, ctx):
    """Where the workspace does not hold the ranges' results, the better of the forms that need none runs: here the one of a
    group of rows a block, whose bits are not those of four groups."""
    kern = rt.kernels("bfloat16")
    rng, bs = np.random.default_rng(D), 16
    pages = ctx // bs
    args = [up(rt, rng.normal(size=s)) for s in ((rows, H * D), (pages, G, bs, D), (pages, G, D, bs))]
    args += [rt.upload(np.array(x, np.int32), "int32") for x in ([list(range(pages))], [0, rows], [ctx])]
    ws = rt.zeros((int(kern.zk_attention_bf16_portion_workspace(rows + 128, H, G, D)) // 4 + 64,), "float32")

    def run(mode, ws_bytes):
        out = rt.zeros((rows, H * D), "bfloat16")
        before = kern.zk_attention_bf16_portion_kernel(mode)
        try:
            kern.zk_attention_bf16(args[0].ptr, H * D, args[1].ptr, args[2].ptr, args[3].ptr, pages, args[4].ptr, args[5].ptr, out.ptr, 1, 1,
                                   rows, ctx, H, G, D, bs, D ** -0.5, 50.0, 0, 0, ws.ptr, ws_bytes, rt.stream)
            return rt.download(out)
        finally:
            kern.zk_attention_bf16_portion_kernel(before)
    group, four, ranges = run(1, 0), run(4, 0), run(5, ws.nbytes)
    assert not np.array_equal(group, four) and not np.array_equal(group, ranges)
    assert np.array_equal(run(0, ws.nbytes), ranges)
    assert np.array_equal(run(0, 0), group) and np.array_equal(run(0, 4096), group)


def test_portions_are_cut_by_their_own_context(rt):
    """Fresh rows beside a decoded request of 3,840 keys: with their own context given, the bits that they have alone."""
    kern = rt.kernels("bfloat16")
    H, G, D, rows, far, bs = 16, 8, 128, 300, 3840, 16
    rng, blocks = np.random.default_rng(7), far // bs
    args = [up(rt, rng.normal(size=s)) for s in ((rows + 1, H * D), (blocks + 19, G, bs, D), (blocks + 19, G, D, bs))]
    table = np.full((2, blocks), -1)
    table[0, :19], table[1] = np.arange(19), 19 + np.arange(blocks)
    args += [rt.upload(np.array(x, np.int32), "int32") for x in (table, [0, rows, rows + 1], [rows, far])]
    n_ws = kern.zk_attention_bf16_portion_workspace(rows + 128, H, G, D) + kern.zk_attention_bf16_workspace(1, H, D, far) + 1024
    ws = rt.zeros((int(n_ws) // 4,), "float32")

    def run(R, max_ctx, portion_ctx):
        out = rt.zeros((rows + 1, H * D), "bfloat16")
        kern.zk_attention_bf16_step(args[0].ptr, H * D, args[1].ptr, args[2].ptr, args[3].ptr, blocks, args[4].ptr, args[5].ptr, out.ptr, R, 1,
                                    rows, max_ctx, H, G, D, bs, D ** -0.5, 50.0, 0, 0, ws.ptr, ws.nbytes, 0, 0, 0, 0, D, 0, None, None, 0,
                                    portion_ctx, rt.stream)
        return rt.download(out)
    alone, beside, unknown = run(1, rows, 0), run(2, far, rows), run(2, far, 0)
    assert np.array_equal(beside[:rows], alone[:rows])
    assert not np.array_equal(unknown[:rows], alone[:rows])         # ranges, by a context that is not theirs
    assert np.array_equal(beside[rows:], unknown[rows:]) and beside[rows:].any()


def test_the_runner_tells_portions_contexts_from_decoded_ones(rt, monkeypatch, tmp_path):
    from conftest import TINY
    from gpu_util import make_runner
    from zse_amd.engine.runner import StepEntry, StepRunner
    from zse_amd.weights import write_random_model
    name = sorted(TINY)[0]
    write_random_model(str(tmp_path), TINY[name][0], seed=1, dtype="bfloat16")
    runner = make_runner(str(tmp_path), "bfloat16", page_size=16, cache_tokens=2048, max_seqs=3, max_batch_tokens=700, max_model_len=1024)
    seen, forward = [], StepRunner._forward
    monkeypatch.setattr(StepRunner, "_forward", lambda self, ctx, *a, **k: (seen.append((ctx.n_multi, ctx.max_ctx, ctx.portion_ctx)),
                                                                           forward(self, ctx, *a, **k))[1])
    for r in "abc":
        runner.add(r)
    runner.step([StepEntry("a", [1] * 600, [])])
    runner.step([StepEntry("a", [2], [0]), StepEntry("b", [3] * 40, [39])])
    runner.step([StepEntry("a", [2], [0]), StepEntry("b", [3] * 300, [0]), StepEntry("c", [3] * 5, [0])])
    runner.step([StepEntry("a", [2], [0]), StepEntry("b", [3], [0])])
    assert seen == [(1, 768, 768), (1, 768, 256), (2, 768, 512), (0, 768, 0)]


@pytest.mark.parametrize("mode", [0, 4, 5])
@pytest.mark.parametrize("H,G,D,E,shift,before,n", [(8, 4, 128, 128, 1, 100, 300), (8, 8, 256, 256, 2, 0, 333), (16, 4, 128, 256, 1, 37, 290)])
def test_key_heads_that_share_a_value_head(rt, mode, H, G, D, E, shift, before, n):
    """2^shift maps of keys over one value head: key head (v << shift) + m serves map m of v's query heads."""
    kern = rt.kernels("bfloat16")
    bs, ctx, V, maps = 16, before + n, G >> shift, 1 << shift
    pages, g = -(-ctx // bs), H // G
    rng = np.random.default_rng(n)
    q, k, v = (rounded(rng.normal(size=s)) for s in ((n, H, D), (ctx, G, D), (ctx, V, E)))
    kc, vc = np.zeros((pages * bs, G, D), np.float32), np.zeros((pages * bs, V, E), np.float32)
    kc[:ctx], vc[:ctx] = k, v
    args = [up(rt, q.reshape(n, -1)), up(rt, kc.reshape(pages, bs, G, D).swapaxes(1, 2)), up(rt, vc.reshape(pages, bs, V, E).transpose(0, 2, 3, 1))]
    args += [rt.upload(np.array(x, np.int32), "int32") for x in ([list(range(pages))], [0, n], [ctx])]
    out = rt.zeros((n, H * E), "bfloat16")
    ws = rt.zeros((int(kern.zk_attention_bf16_portion_workspace(n + 128, H, G, E)) // 4 + 64,), "float32")
    mode_before = kern.zk_attention_bf16_portion_kernel(mode)
    try:
        assert mode == 0 or form_of(ws.nbytes, 1, n, ctx, H, G, D, E)[::2] == (mode, 1)
        kern.zk_attention_bf16_sized(args[0].ptr, H * D, args[1].ptr, args[2].ptr, args[3].ptr, pages, args[4].ptr, args[5].ptr, out.ptr,
                                     1, 1, n, ctx, H, G, D, bs, D ** -0.5, 30.0, 0, 0, ws.ptr, ws.nbytes, 0, 0, 0, shift, E, 0, rt.stream)
        got = rt.download_f32(out).reshape(n, H, E)
    finally:
        kern.zk_attention_bf16_portion_kernel(mode_before)
    want = np.zeros((n, H, E))
    for h in range(H):
        vh, m = (h >> shift) // g, h & (maps - 1)
        want[:, h] = plain(q[:, h:h + 1].astype(np.float64), k[:, (vh << shift) + m][:, None].astype(np.float64),
                           v[:, vh][:, None].astype(np.float64), before, D ** -0.5, 30.0, 0, 0)[:, 0]
    assert np.abs(got - want).max() < 0.03
    assert np.linalg.norm(got - want) < 4e-3 * np.linalg.norm(want)
