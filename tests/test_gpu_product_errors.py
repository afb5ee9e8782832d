"""The error of products against 64 bits where a cut has few waves a strip: what the chains of the kernels before had, not half as much again."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# the relative error that K in as many chains as before gives, and a tenth more; with one chain a wave 2.7e-7, 1.9e-7, 1.8e-7 and 1.9e-7
@pytest.mark.parametrize("kind,N,K,rows,bound", [("head", 65536, 2048, (17, 64), 2.05e-7), ("reader", 4608, 8192, (1, 16), 1.22e-7),
                                                 ("gated", 12800, 1024, (8, 16), 1.55e-7), ("gated", 2048, 4096, (17, 24), 1.65e-7)])
def test_error(kind, N, K, rows, bound):
    from zse_amd.runtime.device import Runtime
    from zse_amd.weights.safetensors import bf16_bits_to_f32, f32_to_bf16_bits
    rt = Runtime.get()
    k = rt.kernels("bfloat16")
    rng = np.random.default_rng(N + K)
    gated = kind == "gated"
    bits = lambda *shape: f32_to_bf16_bits(rng.standard_normal(shape, dtype=np.float32))
    a, w = bits(max(rows), K), bits(N * (2 if gated else 1), K)
    A, W = rt.upload(a, "bfloat16"), rt.upload(w, "bfloat16")
    S = rt.empty((-(-len(w) // 16) * 16, K), "bfloat16")
    k.zk_strip_layout(W.ptr, S.ptr, len(w), K, rt.stream)
    ws = rt.zeros((k.zk_gemm_bf16_workspace() // 4,), "float32")
    z = bf16_bits_to_f32(a).astype(np.float64) @ bf16_bits_to_f32(w).astype(np.float64).T
    want = np.maximum(z[:, :N], 0) * z[:, N:] if gated else z
    for M in rows:
        parts = ctypes.c_int(0)
        C = rt.zeros((M, N), "bfloat16" if kind == "reader" else "float32")
        k.zk_gemm_bf16(A.ptr, K, S.ptr, C.ptr, N, int(kind != "reader"), M, N, K, 5 if gated else 0, 0.0, 1, ws.ptr, ws.nbytes,
                       ctypes.byref(parts) if kind == "reader" else None, rt.stream)
        got = rt.download(C)
        if kind == "reader":
            planes = rt.download(ws)[:parts.value * M * N].reshape(parts.value, M, N)
            got = planes[0]
            for plane in planes[1:]:
                got = got + plane
        assert np.linalg.norm(got - want[:M]) < bound * np.linalg.norm(want[:M]), M
