"""Which kernel or layout a launch takes (host code: no GPU needed), at sizes on both sides of each line."""
import ctypes as C

import pytest


def library(name="kernels_bf16"):
    from zse_amd.runtime import build
    return C.CDLL(build.ensure(name))


# rows, requests, the longest, channels: runs numbered through all requests only where many blocks would find none
@pytest.mark.parametrize("T,R,longest,channels,by_piece", [
    (1, 1, 1, 2048, 0), (200, 200, 1, 8192, 0), (900, 300, 3, 512, 0), (2048, 1, 2048, 2048, 0), (2048, 4, 512, 2048, 0),
    (9000, 1000, 9, 256, 0), (105, 7, 99, 256, 0), (708, 9, 700, 2048, 1), (2500, 501, 2000, 256, 1), (320, 21, 300, 2048, 1)])
def test_runs_of_the_short_convolution(T, R, longest, channels, by_piece):
    """One prompt of 2,048 rows took 12.9 us with its runs looked up and asked for at once, 10.2 without."""
    assert library().zk_conv_rows_by_piece(T, R, longest, channels, 8) == by_piece


# tokens, heads, key heads, channels of a head, values transposed, planes of partial sums; by token in 16 and in 32 bits
@pytest.mark.parametrize("T,nh,nkv,hd,transposed,sums,by_token", [
    (64, 8, 4, 256, 1, 0, (0, 0)), (140, 8, 4, 256, 1, 0, (0, 0)), (200, 8, 4, 256, 1, 0, (0, 1)), (400, 8, 4, 256, 1, 0, (1, 1)),
    (100, 32, 16, 128, 1, 0, (0, 1)), (200, 32, 16, 128, 1, 0, (1, 1)), (200, 16, 4, 64, 1, 0, (0, 0)), (400, 16, 4, 64, 1, 0, (1, 1)),
    (400, 8, 2, 64, 1, 0, (0, 0)), (200, 64, 8, 64, 1, 0, (1, 1)), (400, 64, 8, 32, 1, 0, (1, 1)), (2048, 16, 4, 16, 1, 0, (1, 1)),
    (400, 8, 4, 256, 1, 3, (0, 0)), (1200, 8, 4, 256, 1, 3, (1, 1)), (140, 64, 8, 64, 1, 3, (0, 0)), (400, 64, 8, 64, 1, 3, (1, 1)),
    (64, 32, 16, 128, 0, 0, (0, 0)), (200, 32, 16, 128, 0, 0, (1, 1)), (140, 8, 4, 256, 0, 0, (0, 0)), (400, 8, 4, 256, 0, 3, (1, 1)),
    (100, 16, 4, 16, 0, 0, (0, 0)), (400, 16, 4, 16, 0, 0, (1, 1)), (2048, 4, 2, 16, 0, 0, (1, 1))])
def test_rotation_by_token(T, nh, nkv, hd, transposed, sums, by_token):
    """64 tokens of 32 heads and 2 x 16 of 128 with values in rows take 3.5 us per (token, head) and 4.6 by token, 2,048 of 16 and
    2 x 4 of 16, transposed, 13.9 and 7.2."""
    for name, want in zip(("kernels_bf16", "kernels_f32"), by_token):
        lib = library(name)
        assert lib.zk_rope_by_token(T, nh, nkv, hd, hd, transposed, sums) == want, name
        assert lib.zk_rope_by_token(T, nh, nkv, hd, hd // 2, transposed, sums) == 0      # a part of the head turned: per head


@pytest.mark.parametrize("D,tokens", [(64, 64), (128, 64), (192, 64), (200, 32), (224, 32), (256, 32)])
def test_chunks_of_the_matrix_memory(D, tokens):
    """Chunks of 64 tokens of heads of 256 key channels took 64 us, of 32 52 (600 tokens, four heads of 40 value channels)."""
    floats = library().zk_mlstm_scan_floats
    floats.restype = C.c_size_t
    chunks = lambda L: (600 + L - 1) // L + 2
    assert floats(600, 2, 4, D, 40, 500) == chunks(tokens) * 4 * (D * 40 + D + 3)
    assert floats(600, 2, 4, D, 40, 30) == chunks(32) * 4 * (D * 40 + D + 3)


# up to 16 rows with three strips a block, 17 to 64 rows in long and short ranges, gated in ranges
@pytest.mark.parametrize("epi,M,N,K", [(0, 1, 3584, 14336), (0, 16, 4608, 36864), (0, 8, 3200, 8192), (0, 17, 2304, 9216), (0, 64, 2304, 2048),
                                       (2, 64, 512, 8192)])
def test_ranges_of_k_need_a_workspace(epi, M, N, K):
    """Ranges of K leave their partial sums in the workspace by 16-byte stores: none, a misaligned one or one too small for two of them leave K whole."""
    cut, mid_cut = (C.c_int * 4)(), library().zk_gemm_bf16_mid_cut
    mid_cut.argtypes = [C.c_int] * 5 + [C.c_void_p, C.c_size_t, C.POINTER(C.c_int)]

    def ranges(ws, room, by_reader=1):
        assert mid_cut(epi, by_reader, M, N, K, ws, room, cut) == 1
        return cut[3]

    plane = (2 if epi else 1) * M * -(-N // 16) * 16 * 4
    assert ranges(4096, 320 << 20) > 1
    assert ranges(4096, 2 * plane) == 2
    for ws, room in ((None, 320 << 20), (None, 0), (4096 + 4, 320 << 20), (4096 + 8, 320 << 20), (4096, 2 * plane - 1), (4096, 0)):
        assert ranges(ws, room) == 1, (ws, room)
    if M > 16:
        assert ranges(4096, 320 << 20, 0) > 1 and ranges(None, 320 << 20, 0) == 1


# query heads, key heads, channels of a key and a value, page, pages of a table, values shared by 2^shift key heads; whether they go past the caches
@pytest.mark.parametrize("nh,nkv,hd,vd,bs,table,shift,past", [
    (8, 4, 256, 256, 16, 64, 0, 1), (8, 4, 256, 256, 32, 32, 0, 1), (8, 4, 256, 256, 64, 16, 0, 0), (8, 4, 256, 256, 16, 512, 0, 1),
    (8, 4, 256, 256, 32, 256, 0, 0), (32, 16, 128, 128, 4, 2048, 0, 1), (32, 16, 128, 128, 128, 64, 0, 0), (16, 8, 64, 128, 16, 64, 1, 0)])
def test_values_past_the_caches(nh, nkv, hd, vd, bs, table, shift, past):
    """Where loads past the caches take a line by halves they lose: 64 requests of 4,000 keys, pages of 64 206 and 239 us, of 128 231 and 279; values of two
    key heads 113 and 128."""
    choice = library().zk_attention_bf16_values_past_caches
    assert choice(1, nh, nkv, hd, vd, bs, table, 64, shift) == past
    assert choice(0, nh, nkv, hd, vd, bs, table, 64, shift) == 0


def test_steps_that_pass_through_more_than_the_cache():
    from types import SimpleNamespace as S
    from zse_amd.parts.ops import values_once
    own, step = S(shared=False, lent=False), lambda **kw: S(**{**dict(weights_read_once=False, R=8, max_ctx=1000, cache_token_bytes=24576), **kw})
    assert values_once(step(), own) == 0                                  # 8 x 1,000 x 24 KB: 197 MB
    assert values_once(step(max_ctx=1500), own) == 1
    assert values_once(step(weights_read_once=True), own) == 1
    for other in (S(shared=True, lent=False), S(shared=False, lent=True)):      # the same values are read again within the step
        assert values_once(step(weights_read_once=True), other) == 0


# 32-bit products: tiles of 64 x 32 and 80 x 64 only where K is in whole steps of 32 (else they go through scratch memory), and not for the shortest K
@pytest.mark.parametrize("M,N,K,tile", [(303, 8192, 1024, (80, 64)), (303, 8192, 1000, (64, 64)), (303, 8192, 1023, (64, 64)), (64, 8192, 1024, (64, 32)),
                                        (64, 8192, 1000, (32, 32)), (128, 18432, 520, (32, 32)), (160, 2048, 512, (48, 32)), (150, 18432, 512, (32, 32))])
def test_tiles_of_32_bit_products(M, N, K, tile):
    """128 x 18,432 columns of K 520 took 36.8 us by 32 x 32 and 58.4 by 64 x 32, 160 x 2,048 of 512 10.0 by 48 x 32 and 11.5 by 64 x 32."""
    rows, columns = C.c_int(), C.c_int()
    assert library("kernels_f32").zk_gemm_plain_tile(M, N, K, C.byref(rows), C.byref(columns)) == 1
    assert (rows.value, columns.value) == tile
    assert K % 32 == 0 or tile not in ((64, 32), (80, 64))


@pytest.mark.parametrize("T,H,wide", [
    (1, 2048, 1), (256, 2048, 1), (257, 2048, 0), (512, 2304, 1), (513, 2304, 0), (4096, 2560, 0), (384, 2816, 1), (512, 2816, 0), (1024, 2816, 0),
    (2048, 3072, 0), (512, 3584, 1), (768, 3584, 0), (1024, 3584, 1), (4096, 4096, 1), (256, 4608, 1), (257, 5120, 0), (1024, 5120, 1),
    (512, 8192, 1), (2048, 8192, 1), (64, 1024, 0), (64, 8196, 0), (64, 2050, 0)])
def test_norms_by_1024_threads(T, H, wide):
    """2,048 rows of 3,072 values took 12.1 us by 256 threads and 15.3 by 1,024, 1,024 of 2,816 7.9 and 9.3, 320 of 5,120 as three planes 10.0 and 10.5."""
    assert library().zk_norm_wide(T, H) == wide
    assert library("kernels_f32").zk_norm_wide(T, H) == 0


# strips of gate (and as many of up), rows; strips a block, waves a strip, steps a chunk
@pytest.mark.parametrize("strips,M,cut", [(1, 17, (1, 8, 8)), (256, 64, (1, 8, 8)), (257, 17, (2, 4, 8)), (512, 64, (2, 4, 8)), (513, 1, (3, 4, 4)),
                                          (768, 16, (3, 4, 4)), (769, 1, (4, 2, 4)), (1025, 64, (3, 4, 4)), (1152, 64, (3, 4, 4)), (1280, 17, (3, 4, 4)),
                                          (1537, 64, (4, 2, 4)), (1792, 64, (4, 2, 4)), (2304, 64, (3, 4, 4)), (2560, 33, (2, 4, 8))])
def test_blocks_of_gated_products(strips, M, cut):
    """1,152 strips of K 3,072 at 64 rows took 54.9 us by two waves a strip, 68.6 by one strip a block and 48.8 by three; 1,792 71.8, 102.1 and, by four, 61.1."""
    out = (C.c_int * 4)()
    mid_cut = library().zk_gemm_bf16_mid_cut
    mid_cut.argtypes = [C.c_int] * 5 + [C.c_void_p, C.c_size_t, C.POINTER(C.c_int)]
    assert mid_cut(2, 0, M, 16 * strips, 3072, 4096, 320 << 20, out) == 1
    assert tuple(out) == cut + (1,)


def test_cuts_of_up_to_16_rows():
    """Every product of up to 16 rows that the blocks of gemm_mid_kernel take has one of the four cuts that are built for so few."""
    out = (C.c_int * 4)()
    mid_cut = library().zk_gemm_bf16_mid_cut
    mid_cut.argtypes = [C.c_int] * 5 + [C.c_void_p, C.c_size_t, C.POINTER(C.c_int)]
    seen = set()
    for epi, by_reader in ((0, 0), (0, 1), (1, 0), (4, 0), (2, 0)):
        for strips in [*range(1, 1100), 1536, 2304, 4095, 4096, 16000]:
            for K in (32, 96, 1024, 2048, 2304, 4096, 8192, 14336):
                for M in (1, 16):
                    if mid_cut(epi, by_reader, M, 16 * strips, K, 4096, 320 << 20, out):
                        seen.add((epi == 2,) + tuple(out)[:3])
    assert seen == {(True, 3, 4, 4), (True, 4, 2, 4), (False, 2, 8, 16), (False, 3, 4, 8)}


@pytest.mark.parametrize("strips,M,cut", [(1023, 17, (4, 2, 8)), (1024, 17, (4, 4, 4)), (1025, 17, (3, 4, 4)), (1536, 64, (3, 4, 4)), (1537, 48, (4, 2, 8)),
                                          (1537, 49, (4, 4, 4)), (4095, 17, (4, 2, 8)), (4096, 17, (8, 1, 4)), (1024, 16, (2, 8, 16)), (16000, 1, (2, 8, 16))])
def test_blocks_of_wide_products(strips, M, cut):
    """1,152 strips of K 4,096 took 34.5 us at 32 rows by two waves a strip, 36.9 by four of four strips and 29.7 of three; 2,560 at 17 rows 69.0, 73.8 and, by
    two waves a strip, 62.1."""
    out = (C.c_int * 4)()
    mid_cut = library().zk_gemm_bf16_mid_cut
    mid_cut.argtypes = [C.c_int] * 5 + [C.c_void_p, C.c_size_t, C.POINTER(C.c_int)]
    assert mid_cut(0, 0, M, 16 * strips, 4096, 4096, 320 << 20, out) == 1
    assert tuple(out)[:3] == cut


@pytest.mark.parametrize("strips,K,blocks", [(192, 8192, 0), (193, 8192, 1), (384, 8192, 1), (400, 8192, 0), (400, 11008, 0), (400, 14336, 1), (511, 14336, 1),
                                             (512, 14336, 0), (512, 28672, 0), (513, 8192, 1), (768, 11008, 1), (769, 8192, 0), (832, 14336, 0),
                                             (1023, 28672, 0), (1024, 8192, 1), (288, 8160, 0)])
def test_few_rows_of_long_products(strips, K, blocks):
    """400 strips of K 8,192 took 19.6 us straight from memory and 21.6 by blocks that share the row, 512 of 28,672 80.8 and 82.8 (8 rows 81.2 and 86.3)."""
    out = (C.c_int * 4)()
    mid_cut = library().zk_gemm_bf16_mid_cut
    mid_cut.argtypes = [C.c_int] * 5 + [C.c_void_p, C.c_size_t, C.POINTER(C.c_int)]
    for M in (1, 16):
        assert mid_cut(0, 1, M, 16 * strips, K, 4096, 320 << 20, out) == blocks


@pytest.mark.parametrize("strips,K,blocks", [(512, 2304, 0), (513, 2304, 1), (800, 4096, 1), (801, 4096, 0), (896, 3584, 1), (896, 4096, 0), (960, 2048, 1),
                                             (961, 2048, 0), (1024, 3072, 0)])
def test_few_rows_of_gated_products(strips, K, blocks):
    """1,024 strips of K 4,096 took 48.0 us at one row straight from memory and 50.2 by blocks, 896 42.0 and 44.5."""
    out = (C.c_int * 4)()
    mid_cut = library().zk_gemm_bf16_mid_cut
    mid_cut.argtypes = [C.c_int] * 5 + [C.c_void_p, C.c_size_t, C.POINTER(C.c_int)]
    for M in (1, 16):
        assert mid_cut(2, 0, M, 16 * strips, K, None, 0, out) == blocks


# strips, K, planes of partial sums; whether the gated, the rotating product makes the row in front of it
@pytest.mark.parametrize("strips,K,planes,gated,rotating", [
    (256, 2304, 6, 1, 1), (288, 2304, 4, 1, 1), (288, 2304, 5, 0, 0), (511, 4096, 4, 1, 1), (512, 4096, 6, 1, 1), (576, 2304, 0, 1, 1), (576, 2304, 1, 1, 0),
    (576, 3072, 0, 0, 1), (576, 3584, 0, 1, 1), (576, 3840, 0, 0, 1), (640, 2048, 1, 1, 0), (896, 2048, 0, 1, 1), (896, 3584, 0, 0, 1), (896, 4096, 1, 0, 0),
    (896, 4096, 0, 1, 1), (1152, 3584, 0, 1, 1), (1152, 3584, 2, 0, 0), (1152, 1024, 6, 1, 1), (576, 1024, 0, 0, 1), (256, 4352, 0, 0, 0),
    (256, 2048 + 32, 0, 0, 0), (256, 2304, 7, 0, 0)])
def test_norms_inside_products(strips, K, planes, gated, rotating):
    """Gated 896 strips of K 3,584 took 36.0 us as two launches and 38.8 as one, 640 rotating ones of K 2,304 with four planes 13.7 and 15.4."""
    lib = library()
    assert bool(lib.zk_norm_product_supports(16 * strips, K, planes)) == gated
    assert bool(lib.zk_norm_rope_product_supports(16 * strips, K, planes)) == rotating


# rows, columns, K, channels of a head
@pytest.mark.parametrize("M,N,K,hd,pays", [(17, 1536, 2560, 128, 1), (17, 1536, 3072, 128, 0), (64, 4096, 2304, 256, 1), (64, 4096, 3584, 256, 1),
                                           (64, 4096, 4096, 256, 0), (64, 6144, 4096, 128, 1), (17, 6144, 4608, 128, 0), (64, 8192, 3584, 256, 1),
                                           (64, 8192, 4608, 128, 1), (64, 8192, 5120, 128, 0), (32, 10240, 2304, 128, 1), (33, 10240, 512, 128, 0),
                                           (17, 10240, 4096, 256, 0)])
def test_rotating_products_of_17_to_64_rows(M, N, K, hd, pays):
    """1,536 columns of K 4,096 took 11.1 and 13.7 us at 17 and 64 rows as two launches, 12.7 and 17.4 as one; 10,240 of 4,096 at 64 26.8 and 35.6."""
    lib = library()
    assert lib.zk_qkv_rope_rows_bf16_pays(M, N, K, hd) == pays
    assert lib.zk_qkv_rope_rows_bf16_supports(M, K, hd, hd) == 1        # what it can do is another matter
