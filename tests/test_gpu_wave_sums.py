"""Sums and maxima over waves and blocks of common.h where lanes are missing: a block that is not whole waves, lanes
left out by a condition.  An extension's kernel may call them so."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def dev():
    import toy_kernels  # noqa: F401  (registers zk_toy_sums)
    from zse_amd.runtime.device import Runtime
    rt = Runtime.get()
    return rt, rt.kernels("float32")


@pytest.mark.parametrize("n", [1, 15, 31, 32, 33, 63, 64, 65, 100, 127, 512, 1000, 1024])
def test_blocks_of_any_size(n):
    rt, k = dev()
    v = np.random.default_rng(n).normal(size=n).astype(np.float32) - 3      # (all below zero: a lane that counts as 0 shows in the maximum)
    out = rt.zeros((4, n), "float32")
    V = rt.upload(v)
    k.zk_toy_sums(V.ptr, out.ptr, n, 0, rt.stream)
    got = rt.download(out)
    for w in range(0, n, 64):
        wave = v[w:w + 64]
        # 64 float additions at most
        assert np.abs(got[0, w:w + 64] - wave.astype(np.float64).sum()).max() <= 64 * 2.0 ** -24 * np.abs(wave).sum()
        assert (got[1, w:w + 64] == wave.max()).all()
    assert np.abs(got[2] - v.astype(np.float64).sum()).max() <= 80 * 2.0 ** -24 * np.abs(v).sum()
    assert (got[2] == got[2, 0]).all() and (got[3] == n).all()


@pytest.mark.parametrize("n", [1, 4, 34, 64])
def test_some_lanes_of_a_wave(n):
    rt, k = dev()
    v = np.random.default_rng(n).normal(size=n).astype(np.float32) - 3
    out = rt.zeros((4, n), "float32")
    V = rt.upload(v)
    k.zk_toy_sums(V.ptr, out.ptr, n, 1, rt.stream)
    got, there = rt.download(out), v[::3]
    assert np.abs(got[0, ::3] - there.astype(np.float64).sum()).max() <= 64 * 2.0 ** -24 * np.abs(there).sum()
    assert (got[1, ::3] == there.max()).all()
