"""Products that read their weights past the caches: the same bits as through them, in every kernel that a step of a large model takes."""
import ctypes

import numpy as np
import pytest

from test_gpu_mid_products import setup

pytestmark = pytest.mark.gpu


# K in ranges left to the reader and joined by a launch: a strip a block (few long ones), three, four in short and in long ranges
@pytest.mark.parametrize("N,K,rows", [(1024, 4096, (1, 16)), (4608, 4096, (1, 16)), (3200, 8192, (1, 7, 16)), (2304, 2048, (17, 48, 64)), (2048, 8192, (17, 33, 64))])
def test_ranges(N, K, rows):
    rt, k, A, S, ws, want = setup(N, K, N, N + K)
    for M in rows:
        seen = []
        for once in (1, 3):
            parts = ctypes.c_int(0)
            C = rt.zeros((M, N), "bfloat16")
            k.zk_gemm_bf16(A.ptr, K, S.ptr, C.ptr, N, 0, M, N, K, 0, 0.0, once, ws.ptr, ws.nbytes, ctypes.byref(parts), rt.stream)
            assert parts.value > 1
            planes = rt.download(ws)[:parts.value * M * N].reshape(parts.value, M, N).copy()
            # float sums of K products of size K^-0.5, in another order
            assert np.abs(planes.astype(np.float64).sum(0) - want[:M]).max() < 2e-5 * np.abs(want).max()
            k.zk_gemm_bf16(A.ptr, K, S.ptr, C.ptr, N, 0, M, N, K, 0, 0.0, once, ws.ptr, ws.nbytes, None, rt.stream)
            seen.append((planes, rt.download(C)))
        assert all(np.array_equal(a, b) for a, b in zip(*seen)), M


@pytest.mark.parametrize("nh,nkv,hd,K", [(8, 4, 256, 2304), (33, 15, 96, 160)])
@pytest.mark.parametrize("M", [1, 16, 17, 40, 64])
def test_rotating(M, nh, nkv, hd, K):
    from zse_amd.runtime.device import Runtime
    from zse_amd.weights.safetensors import f32_to_bf16_bits
    rt = Runtime.get()
    k = rt.kernels("bfloat16")
    rng = np.random.default_rng(M + hd + K)
    N, bs, pages = (nh + 2 * nkv) * hd, 8, 12
    up = lambda x: rt.upload(f32_to_bf16_bits(np.ascontiguousarray(x, np.float32)), "bfloat16")
    A, W, S = up(rng.normal(size=(M, K))), up(rng.normal(size=(N, K)) * K ** -0.5), rt.empty((N, K), "bfloat16")
    k.zk_strip_layout(W.ptr, S.ptr, N, K, rt.stream)
    pos, slots = rt.upload(rng.integers(0, 8000, M).astype(np.int32)), rt.upload(rng.permutation(pages * bs)[:M].astype(np.int32))
    freq = rt.upload((10000.0 ** (-np.arange(hd // 2) * 2 / hd)).astype(np.float32))
    seen = []
    for once in (1, 3):
        Q, kc, vc = rt.zeros((M, N), "bfloat16"), rt.zeros((pages * bs * nkv * hd,), "bfloat16"), rt.zeros((pages * bs * nkv * hd,), "bfloat16")
        run = k.zk_qkv_rope_bf16 if M <= 16 else k.zk_qkv_rope_rows_bf16
        run(A.ptr, K, S.ptr, Q.ptr, N, M, K, once, pos.ptr, slots.ptr, freq.ptr, kc.ptr, vc.ptr, nh, nkv, hd, bs, 1, rt.stream)
        seen.append([rt.download(t) for t in (Q, kc, vc)])
    assert all(np.array_equal(a, b) for a, b in zip(*seen)) and all(x.any() for x in seen[0])
