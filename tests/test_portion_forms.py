"""Which kernel a launch of portions takes (host code: no GPU needed)."""
import ctypes as C

import pytest


def form_of(room, R, rows, ctx, H, G, D, E=0, bs=16, window=0, chunk=0, keep=0, wide_weights=0, not_theirs=0):
    """(groups of rows a block, or 5 for four with the keys in ranges; tiles of a range; by attn_stream_kernel)"""
    from zse_amd.runtime import build
    lib = C.CDLL(build.ensure("kernels_bf16"))
    ranges, stream = C.c_int(-1), C.c_int(-1)
    form = lib.zk_attention_bf16_portion_form(R, rows, ctx, not_theirs, H, G, D, E or D, bs, window, chunk, keep, wide_weights,
                                              C.c_size_t(room), C.byref(ranges), C.byref(stream))
    return form, ranges.value, stream.value


# requests, rows, context, heads, key heads, channels; the form without ranges
CASES = [((1, 512, 4096, 8, 4, 256), 1), ((1, 512, 4096, 32, 16, 128), 1), ((1, 1024, 2048, 8, 4, 256), 1),
         ((2, 1024, 3000, 8, 4, 256), 4), ((1, 3000, 4096, 8, 4, 256), 4)]


@pytest.mark.parametrize("case,whole", CASES)
def test_without_room_for_ranges_the_better_form_that_needs_none(case, whole):
    form, tiles, stream = form_of(1 << 30, *case)
    assert (form, stream) == (5, 1) and tiles > 0
    assert form_of(0, *case)[0] in ((1, 2) if whole == 1 else (4,))
    assert form_of(4096, *case) == form_of(0, *case)


def test_pages_whose_places_32_bits_do_not_hold():
    assert form_of(0, 1, 4000, 4000, 8, 4, 256, bs=1 << 23)[2] == 1
    assert form_of(0, 1, 4000, 4000, 8, 4, 256, bs=1 << 24)[2] == 0
    assert form_of(0, 1, 4000, 4000, 8, 4, 256, bs=8)[2] == 0
    assert form_of(0, 1, 4000, 4000, 8, 4, 256, wide_weights=1)[2] == 0


@pytest.mark.parametrize("case,form", [((1, 2048, 2048, 32, 16, 128), 4), ((1, 2048, 2048, 32, 8, 128), 4), ((1, 2048, 2048, 16, 8, 256), 4),
                                       ((1, 104, 104, 8, 8, 128), 1), ((2, 116, 116, 8, 8, 128), 1)])
def test_launches_that_a_form_with_fewer_blocks_runs_faster(case, form):
    """Two ranges a block of rows lie on halves of the chip that have unlike work, and a block of four groups that has rows for
    one is slower than a group a block (94 us against 70, 80 against 61, 98 against 81, 12.4 against 10.5 twice)."""
    assert form_of(1 << 30, *case)[0] == form


@pytest.mark.parametrize("R,rows,H,G,D", [(8, 128, 32, 16, 128), (4, 512, 16, 4, 128), (1, 2048, 16, 4, 128), (1, 1024, 32, 16, 128)])
def test_many_groups_beside_a_long_decoded_context(R, rows, H, G, D):
    """A context that may be a decoded request's does not cut the keys of many groups into ranges."""
    assert form_of(1 << 30, R, rows, 8192, H, G, D)[0] == 5
    assert form_of(1 << 30, R, rows, 8192, H, G, D, not_theirs=1)[0] == 4


# requests, rows, context, heads, key heads, channels, chunk: the beginning of a chunk among the rows, at their end, in front of them, in front
# of the last one
@pytest.mark.parametrize("case,short", [((1, 512, 8448, 8, 4, 256, 8192), 0), ((1, 256, 8208, 32, 16, 128, 8192), 0),
                                        ((1, 256, 8192, 32, 16, 128, 8192), 0), ((1, 64, 8193, 8, 2, 128, 8192), 0),
                                        ((3, 64, 8200, 16, 4, 128, 8192), 0), ((1, 256, 8448, 8, 4, 256, 8192), 1),
                                        ((1, 64, 8256, 32, 16, 128, 8192), 1), ((1, 64, 100, 32, 16, 128, 64), 1),
                                        ((1, 512, 8448, 8, 4, 256, 128), 1)])
def test_a_chunk_that_begins_among_the_rows(case, short):
    """The rows in front of it see the whole chunk before: their block has the most keys, not the last one."""
    R, rows, ctx, H, G, D, chunk = case
    assert (form_of(1 << 30, R, rows, ctx, H, G, D, chunk=chunk)[2] == 2) == bool(short)


# requests, rows, context, heads, key heads, channels, window: many requests whose keys several blocks fetch, with long contexts and short
# ones, and one block for all rows of a request
@pytest.mark.parametrize("case,short", [((16, 16, 1516, 32, 16, 128, 0), 0), ((16, 16, 416, 32, 8, 128, 0), 0), ((8, 33, 233, 32, 16, 128, 0), 0),
                                        ((8, 17, 417, 64, 8, 128, 300), 0), ((16, 16, 76, 32, 8, 128, 0), 1),
                                        ((12, 37, 137, 8, 4, 256, 0), 1), ((64, 4, 404, 32, 8, 128, 0), 1), ((1, 150, 650, 32, 16, 128, 0), 1)])
def test_few_rows_of_many_requests(case, short):
    """Memory bounds them where blocks of 16 rows fetch a request's keys several times: 16 of 16 rows behind 1,500 keys, 32 heads over
    16 of 128, took 60.6 us in place of 48.2."""
    R, rows, ctx, H, G, D, window = case
    assert (form_of(1 << 30, R, rows, ctx, H, G, D, window=window)[2] == 2) == bool(short)
