"""Decoded tokens' attention over few and many parts: the same bits where the sums are the same."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def dev():
    from zse_amd.runtime.device import Runtime
    rt = Runtime.get()
    return rt, rt.kernels("bfloat16")


@pytest.mark.parametrize("nh,nkv,hd", [(8, 4, 256), (8, 2, 128), (16, 1, 64)])
def test_attention_of_few_and_many_blocks_and_with_a_window_that_shows_all(nh, nkv, hd):
    """Requests of one to 78 parts of 128 keys: alone, among so many that the chip is full,
    and behind a window as long as the longest context, whose parts are counted from the request's length: the same bits."""
    from zse_amd.weights.safetensors import f32_to_bf16_bits
    rt, k = dev()
    rng = np.random.default_rng(hd)
    up = lambda x: rt.upload(f32_to_bf16_bits(np.ascontiguousarray(x, np.float32)), "bfloat16")
    bs, lens = 16, [1, 128, 129, 1000, 1030, 2049, 4100, 9900]
    ends = np.cumsum([0] + [-(-n // bs) for n in lens])
    kc, vc = up(rng.normal(size=(ends[-1], nkv, bs, hd))), up(rng.normal(size=(ends[-1], nkv, hd, bs)))
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
    for copies, window in ((1, 9983), (12, 0), (12, 9900)):
        got = run(copies, window, 32)
        assert all(np.array_equal(x, want) for x in got), (copies, window)
