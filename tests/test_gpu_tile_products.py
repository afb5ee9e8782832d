"""Products of more than 64 rows by weights in strips: every tile shape, whole, with K in ranges
(joined by a launch or handed to the reader) and with the last round's tiles in ranges, at sizes whose
last rows and columns are not full, and every way out (16 or 32 bits, rows of any length and
distance, each epilogue)."""
import ctypes as C
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# tile (its number in tile_shapes), ranges of K, ranges of the last round, gated, rows, columns, K
CUTS = [
    (0, 1, 1, 0, 1031, 10960, 128), (0, 1, 1, 1, 409, 12304, 128), (1, 1, 1, 0, 546, 11232, 768), (1, 1, 1, 1, 300, 9088, 768),
    (1, 3, 1, 1, 518, 1824, 3072), (1, 1, 8, 1, 328, 11136, 2112), (2, 1, 1, 0, 693, 8240, 576), (2, 1, 1, 1, 199, 11152, 576),
    (2, 3, 1, 0, 776, 2496, 3072), (2, 3, 1, 1, 2049, 464, 3072), (2, 1, 8, 0, 661, 10960, 2112), (3, 1, 1, 0, 719, 11184, 64),
    (3, 1, 1, 1, 338, 11216, 64), (4, 1, 1, 0, 332, 10992, 512), (4, 1, 1, 1, 129, 11392, 512), (4, 2, 1, 1, 352, 2704, 3072),
    (5, 1, 1, 0, 129, 11088, 512), (5, 1, 1, 1, 140, 5584, 512), (5, 5, 1, 0, 3078, 144, 3072), (5, 5, 1, 1, 2961, 80, 3072),
    (6, 1, 1, 0, 454, 8304, 64), (6, 1, 1, 1, 204, 8400, 64), (6, 1, 8, 1, 1802, 2192, 2112), (7, 1, 1, 0, 386, 9776, 320),
    (7, 1, 1, 1, 143, 11072, 320), (7, 3, 1, 0, 261, 6816, 3072), (8, 1, 1, 0, 272, 11760, 768), (8, 1, 1, 1, 69, 8368, 768),
    (9, 1, 1, 0, 65, 32, 64), (9, 1, 1, 1, 65, 32, 64), (9, 4, 1, 0, 66, 32, 1024), (9, 4, 1, 1, 66, 32, 1024),
]

# gated, 256 x 256 tiles in whole rounds and the columns behind them by another tile: that tile, rows, columns, K
RESTS = [(1, 1545, 11664, 576), (2, 1538, 11360, 576), (3, 1031, 10912, 1536), (4, 1415, 12320, 576), (5, 675, 12368, 1024),
         (7, 1415, 12944, 576), (8, 1057, 8368, 1024), (9, 642, 12336, 2112)]


@pytest.fixture(scope="module")
def rt():
    from zse_amd.runtime.device import Runtime
    return Runtime.get()


def cut_of(gated, by_reader, M, N, K):
    from zse_amd.runtime import build
    out = [C.c_int() for _ in range(4)]
    assert C.CDLL(build.lib_path("kernels_bf16")).zk_gemm_bf16_tile_cut(gated, by_reader, M, N, K, *map(C.byref, out)) == 0
    return tuple(v.value for v in out)


def operands(rt, M, rows, K, seed):
    """(A, W in strips) on the device and A W^T in 64 bits.  Sums of about size 1."""
    from zse_amd.weights.safetensors import bf16_bits_to_f32, f32_to_bf16_bits
    rng = np.random.default_rng(seed)
    bits = lambda *shape: f32_to_bf16_bits(rng.standard_normal(shape, np.float32) * np.float32(K ** -0.25))
    a, w = bits(M, K), bits(rows, K)
    W, S = rt.upload(w, "bfloat16"), rt.empty((-(-rows // 16) * 16, K), "bfloat16")
    rt.kernels("bfloat16").zk_strip_layout(W.ptr, S.ptr, rows, K, rt.stream)
    rt.sync()
    return rt.upload(a, "bfloat16"), S, bf16_bits_to_f32(a).astype(np.float64) @ bf16_bits_to_f32(w).astype(np.float64).T


def workspace(rt):
    """Scratch that holds NaN, so that a sum nobody wrote shows."""
    n = rt.kernels("bfloat16").zk_gemm_bf16_workspace() // 4
    return rt.upload(np.full(n, np.nan, np.float32), "float32")


def gelu_tanh(z):
    return 0.5 * z * (1 + np.tanh(math.sqrt(2 / math.pi) * (z + 0.044715 * z ** 3)))


@pytest.mark.parametrize("shape,ks,tail,gated,M,N,K", CUTS)
def test_every_cut(rt, shape, ks, tail, gated, M, N, K):
    assert cut_of(gated, 0, M, N, K) == (shape, ks, tail, -1)
    check_product(rt, gated, M, N, K)


@pytest.mark.parametrize("rest,M,N,K", RESTS)
def test_columns_behind_the_whole_rounds(rt, rest, M, N, K):
    assert cut_of(1, 0, M, N, K) == (0, 1, 1, rest)
    check_product(rt, 1, M, N, K)


def check_product(rt, gated, M, N, K):
    A, S, z = operands(rt, M, N * (1 + gated), K, seed=M + N)
    ws = workspace(rt)
    out = rt.upload(np.full((M + 2, N + 8), 0x4040, np.uint16), "bfloat16")
    rt.kernels("bfloat16").zk_gemm_bf16(A.ptr, K, S.ptr, out.ptr, N + 8, 0, M, N, K, 2 if gated else 0, 0.0, 1, ws.ptr, ws.nbytes,
                                        None, rt.stream)
    got = rt.download_f32(out)
    want = gelu_tanh(z[:, :N]) * z[:, N:] if gated else z
    # a result rounded to 8 bits of mantissa; K float additions of products of size K^-0.5
    assert (np.abs(got[:M, :N] - want) <= np.abs(want) * 2.0 ** -8 + 1e-4 * (1 + 3 * gated)).all()
    assert (got[M:] == 3.0).all() and (got[:, N:] == 3.0).all()


@pytest.mark.parametrize("M,N,K", [(535, 2304, 9216), (66, 32, 1024), (261, 6816, 3072), (1000, 1008, 4096)])
def test_sums_for_the_reader(rt, M, N, K):
    """A caller with ``parts`` gets planes that add up to the product."""
    assert cut_of(0, 1, M, N, K)[1] > 1
    A, S, want = operands(rt, M, N, K, seed=M)
    ws, out, parts = workspace(rt), rt.zeros((M, N), "bfloat16"), C.c_int(-1)
    rt.kernels("bfloat16").zk_gemm_bf16(A.ptr, K, S.ptr, out.ptr, N, 0, M, N, K, 0, 0.0, 1, ws.ptr, ws.nbytes, C.byref(parts), rt.stream)
    assert parts.value == cut_of(0, 1, M, N, K)[1]
    from zse_amd.runtime.device import Tensor
    got = rt.download(Tensor(ws.ptr, (parts.value, M, N), "float32", ws.owner)).astype(np.float64).sum(0)
    assert np.abs(got - want).max() <= 1e-4
    assert not rt.download(out).any()


EPILOGUES = {0: lambda z: z, 1: lambda z: 2 * np.tanh(z / 2), 7: lambda z: np.maximum(z, 0) ** 2,
             8: lambda z: 0.5 * z * (1 + np.vectorize(math.erf)(z / math.sqrt(2)))}
GATES = {2: lambda g, u: gelu_tanh(g) * u, 3: lambda g, u: g / (1 + np.exp(-g)) * u, 5: lambda g, u: np.maximum(g, 0) * u,
         6: lambda g, u: np.minimum(g, 2) / (1 + np.exp(-1.702 * np.minimum(g, 2))) * (np.clip(u, -2, 2) + 1)}


@pytest.mark.parametrize("f32", [0, 1])
@pytest.mark.parametrize("M,N,extra", [(130, 203, 0), (97, 200, 4), (300, 136, 8)])       # odd rows, rows of pieces at odd distances, whole pieces
@pytest.mark.parametrize("K", [128, 2048])            # whole, in ranges
@pytest.mark.parametrize("epi", sorted(EPILOGUES) + sorted(GATES))
def test_every_way_out(rt, epi, K, M, N, extra, f32):
    gated = epi in GATES
    if gated:
        N = N // 16 * 16         # gate and up rows are whole strips each
    A, S, z = operands(rt, M, N * (1 + gated), K, seed=epi + K)
    ws = workspace(rt)
    ld = N + extra
    out = rt.upload(np.full((M + 1, ld), 3.0, np.float32) if f32 else np.full((M + 1, ld), 0x4040, np.uint16), "float32" if f32 else "bfloat16")
    rt.kernels("bfloat16").zk_gemm_bf16(A.ptr, K, S.ptr, out.ptr, ld, f32, M, N, K, epi, 2.0, 1, ws.ptr, ws.nbytes, None, rt.stream)
    got = rt.download_f32(out)
    want = GATES[epi](z[:, :N], z[:, N:]) if gated else EPILOGUES[epi](z)
    # 32 bits: a product of two such sums may be ten times their size
    assert (np.abs(got[:M, :N] - want) <= np.abs(want) * (1e-5 if f32 else 2.0 ** -8) + 1e-4 * (1 + 9 * (gated or epi == 7))).all()
    assert (got[M:] == 3.0).all() and (got[:, N:] == 3.0).all()


def test_the_static_array_where_its_sums_do_not_fit(rt):
    """535 x 2304 x 9216: ranges of K whose sums are more than the array's 16 MiB."""
    M, N, K = 535, 2304, 9216
    assert cut_of(0, 0, M, N, K)[1] * M * N * 4 > 16 << 20
    A, S, want = operands(rt, M, N, K, seed=1)
    out = rt.zeros((M, N), "bfloat16")
    from zse_amd.runtime import build
    dll = C.CDLL(build.lib_path("kernels_bf16"))
    VP, I, F = C.c_void_p, C.c_int, C.c_float
    dll.zk_gemm_bf16_static.argtypes = [VP, I, VP, VP, I, I, I, I, I, I, F, I, VP]
    assert dll.zk_gemm_bf16_static(A.ptr, K, S.ptr, out.ptr, N, 0, M, N, K, 0, 0.0, 1, rt.stream) == 0
    got = rt.download_f32(out)
    assert (np.abs(got - want) <= np.abs(want) * 2.0 ** -8 + 1e-4).all()


STATIC = [
    # rows, columns, K, gated: ranges of K, of the last round's tiles, whose sums are more than the static array's 16 MiB
    (535, 2304, 9216, 0), (526, 4099, 4608, 0), (412, 3072, 4608, 1), (583, 2304, 4608, 1), (184, 2304, 18432, 1),
    (2179, 4096, 3072, 0), (583, 8208, 3072, 1), (3604, 2304, 3072, 1), (2863, 3072, 3072, 0),
]


@pytest.mark.parametrize("f32", [0, 1])
@pytest.mark.parametrize("M,N,K,gated", STATIC)
def test_the_static_array_gives_the_bits_of_the_workspace_also_where_the_sums_do_not_fit(rt, M, N, K, gated, f32):
    from zse_amd.runtime import build
    shape, ks, tail_ks, _ = cut_of(gated, 0, M, N, K)
    assert ks > 1 or tail_ks > 1
    if ks > 1:
        assert ks * (1 + gated) * M * -(-N // 16) * 16 * 4 > 16 << 20
    kern, epi, ld = rt.kernels("bfloat16"), 3 if gated else 0, N + 5
    A, S = rt.empty((M, K), "bfloat16"), rt.empty((-(-N * (1 + gated) // 16) * 16, K), "bfloat16")
    for t, seed in ((A, 1), (S, 2)):
        kern.zk_fill_normal(t.ptr, 1, t.numel, seed, 1, 0.0, K ** -0.25, rt.stream)
    dll = C.CDLL(build.lib_path("kernels_bf16"))
    VP, I, F = C.c_void_p, C.c_int, C.c_float
    dll.zk_gemm_bf16_static.argtypes = [VP, I, VP, VP, I, I, I, I, I, I, F, I, VP]
    got, want = (rt.upload(np.full((M, ld), 3.0, np.float32) if f32 else np.full((M, ld), 0x4040, np.uint16), "float32" if f32 else "bfloat16")
                 for _ in range(2))
    ws = workspace(rt)
    kern.zk_gemm_bf16(A.ptr, K, S.ptr, want.ptr, ld, f32, M, N, K, epi, 0.0, 1, ws.ptr, ws.nbytes, None, rt.stream)
    assert dll.zk_gemm_bf16_static(A.ptr, K, S.ptr, got.ptr, ld, f32, M, N, K, epi, 0.0, 1, rt.stream) == 0
    got, want = rt.download(got), rt.download(want)
    assert (want[:, :N] != 0).any() and (want[:, N:] == (3.0 if f32 else 0x4040)).all()
    assert np.array_equal(got, want)


def test_what_the_static_array_refuses_of_weights_in_strips(rt):
    """The shapes that it refused of them before they had tiles of their own: those of weights that lie row by row."""
    from zse_amd.runtime import build
    M, N, K = 1024, 1024, 65536
    A, S, out = rt.zeros((M, K), "bfloat16"), rt.zeros((N, K), "bfloat16"), rt.zeros((M, N), "bfloat16")
    dll = C.CDLL(build.lib_path("kernels_bf16"))
    VP, I, F = C.c_void_p, C.c_int, C.c_float
    dll.zk_gemm_bf16_static.argtypes = [VP, I, VP, VP, I, I, I, I, I, I, F, I, VP]
    dll.zk_last_error.restype = C.c_char_p
    for strip in (0, 1):
        assert dll.zk_gemm_bf16_static(A.ptr, K, S.ptr, out.ptr, N, 0, M, N, K, 0, 0.0, strip, rt.stream) != 0
        assert b"static scratch array holds 16777216" in dll.zk_last_error()
    rt.sync()
