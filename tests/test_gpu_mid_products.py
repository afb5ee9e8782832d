"""Products of up to 64 rows by weights in strips, every cut of their kernel: strips a block, waves a strip, short and long chunks, K shorter than
a chunk or not whole ones, strips and rows that do not fill a block, ranges of K joined by a launch or left to the reader."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def setup(N, K, rows, seed):
    from zse_amd.runtime.device import Runtime
    from zse_amd.weights.safetensors import bf16_bits_to_f32, f32_to_bf16_bits
    rt = Runtime.get()
    k = rt.kernels("bfloat16")
    rng = np.random.default_rng(seed)
    bits = lambda *shape: f32_to_bf16_bits(rng.standard_normal(shape, dtype=np.float32) * np.float32(K ** -0.25))
    a, w = bits(64, K), bits(rows, K)
    A, W = rt.upload(a, "bfloat16"), rt.upload(w, "bfloat16")
    S = rt.empty((-(-rows // 16) * 16, K), "bfloat16")
    k.zk_strip_layout(W.ptr, S.ptr, rows, K, rt.stream)
    ws = rt.zeros((k.zk_gemm_bf16_workspace() // 4,), "float32")
    return rt, k, A, S, ws, bf16_bits_to_f32(a).astype(np.float64) @ bf16_bits_to_f32(w).astype(np.float64).T


# one, two, three and four strips a block, the last block not full; in ranges with a join
@pytest.mark.parametrize("N,K", [(80, 32), (80, 288), (16 * 257, 96), (16 * 511, 160), (16 * 575, 96), (16 * 893, 416), (64, 8192)])
def test_gated(N, K):
    rt, k, A, S, ws, z = setup(N, K, 2 * N, N + K)
    want = np.maximum(z[:, :N], 0) * z[:, N:]
    few = {}
    for M in (1, 9, 16, 17, 33, 48, 49, 64):
        for ldc in (N, N + 3):
            C = rt.upload(np.full((M + 1, ldc), 0x4040, np.uint16), "bfloat16")
            k.zk_gemm_bf16(A.ptr, K, S.ptr, C.ptr, ldc, 0, M, N, K, 5, 0.0, 1 if ldc == N else 3, ws.ptr, ws.nbytes, None, rt.stream)
            got = rt.download_f32(C)
            # a result rounded to 8 bits of mantissa; two float sums of K products of size K^-0.5, each times the other
            assert (np.abs(got[:M, :N] - want[:M]) <= np.abs(want[:M]) * 2.0 ** -8 + 4e-4).all(), (M, ldc)
            assert (got[M:] == 3.0).all() and (got[:, N:] == 3.0).all()
            if M <= 16:
                few.setdefault(0, got[0, :N])
                assert np.array_equal(got[0, :N], few[0])          # a row does not know of the others


# heads of four and eight strips a block with a last strip that is not full, by two strips a block up to 16 rows (K of 2,048)
@pytest.mark.parametrize("N,K", [(16 * 1030 + 5, 64), (16 * 4100 + 11, 96), (16 * 1024 + 1, 2048), (16 * 1030, 2080)])
def test_heads(N, K):
    rt, k, A, S, ws, z = setup(N, K, N, N)
    want = 30.0 * np.tanh(z / 30.0)
    few = {}
    for M in (1, 5, 16, 17, 40, 64):
        for ldc in (N, N + 3):
            C = rt.upload(np.full((M + 1, ldc), 3.0, np.float32))
            k.zk_gemm_bf16(A.ptr, K, S.ptr, C.ptr, ldc, 1, M, N, K, 1, 30.0, 1 if ldc == N else 3, ws.ptr, ws.nbytes, None, rt.stream)
            got = rt.download(C)
            # float sums of K products of size K^-0.5, and the float tanh
            assert np.abs(got[:M, :N] - want[:M]).max() < 2e-5 * np.abs(want).max(), (M, ldc)
            assert (got[M:] == 3.0).all() and (got[:, N:] == 3.0).all()
            if M <= 16:
                few.setdefault(0, got[0, :N])
                assert np.array_equal(got[0, :N], few[0])
        picks, ids = rt.zeros((k.zk_head_pick_bf16_workspace(M, N) // 4,), "float32"), rt.zeros((M,), "int32")
        k.zk_head_pick_bf16(A.ptr, K, S.ptr, M, N, K, 30.0, 1, picks.ptr, picks.nbytes, ids.ptr, rt.stream)
        assert np.array_equal(rt.download(ids), np.argmax(got[:M, :N], 1)), M


# short ranges (chunks of four), long ones; up to 16 rows three strips a block
@pytest.mark.parametrize("N,K,rows", [(2304, 2048, (17, 48, 64)), (1024, 1056, (17, 64)), (2048, 8192, (17, 33, 64)), (3200, 8192, (1, 7, 16, 64))])
def test_ranges(N, K, rows):
    rt, k, A, S, ws, want = setup(N, K, N, N + K)
    few = {}
    for M in rows:
        parts = ctypes.c_int(0)
        C = rt.zeros((M, N), "bfloat16")
        k.zk_gemm_bf16(A.ptr, K, S.ptr, C.ptr, N, 0, M, N, K, 0, 0.0, 1, ws.ptr, ws.nbytes, ctypes.byref(parts), rt.stream)
        P = parts.value
        assert P > 1, M
        planes = rt.download(ws)[:P * M * N].reshape(P, M, N)
        # float sums of K products of size K^-0.5, in another order
        assert np.abs(planes.astype(np.float64).sum(0) - want[:M]).max() < 2e-5 * np.abs(want).max()
        if M <= 16:
            few.setdefault(0, planes[:, 0])
            assert np.array_equal(planes[:, 0], few[0])
        k.zk_gemm_bf16(A.ptr, K, S.ptr, C.ptr, N, 0, M, N, K, 0, 0.0, 1, ws.ptr, ws.nbytes, None, rt.stream)
        got = rt.download_f32(C)
        assert (np.abs(got - want[:M]) <= np.abs(want[:M]) * 2.0 ** -8 + 1e-4).all(), M
