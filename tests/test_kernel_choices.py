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
