"""When a block hands the norm in front of the next product on unmade (host code: no GPU needed)."""
from types import SimpleNamespace

import pytest

from zse_amd.parts.block import Block
from zse_amd.parts.norm import RMSNorm
from zse_amd.parts.ops import PendingNorm
from zse_amd.runtime.device import BF16, F32, Tensor

H, WORKSPACE = 256, 1 << 30


class Kernels:
    def has(self, name):
        return True

    def __getattr__(self, name):
        return lambda *a: None


class Arena:
    """Places in the step's own memory, one after the other; ``base`` is where the next block begins again."""

    def __init__(self):
        self.next = 4096

    def alloc(self, shape, dtype=BF16):
        t = Tensor(self.next, shape, dtype)
        self.next += -(-t.nbytes // 256) * 256
        return t


def norm():
    n = RMSNorm(SimpleNamespace(eps=1e-6, unit_offset=True, size=H))
    n.weight = Tensor(1 << 20, (H,), F32)
    return n


def block(ffn):
    b = Block.__new__(Block)
    b.spec = SimpleNamespace(arrangement="sandwich")
    b.norms = {r: norm() for r in ("pre_mixer", "post_mixer", "pre_ffn", "post_ffn")}
    b.mixer = SimpleNamespace(forward=lambda ctx, x, cache: ctx.alloc((1, H)), takes_pending_norm=lambda ctx, size, planes: True)
    b.ffn = SimpleNamespace(forward=ffn)
    return b


def context(nxt):
    arena = Arena()
    return SimpleNamespace(alloc=arena.alloc, arena=arena, k=Kernels(), dtype=BF16, tuned=True, stream=0, next_block=nxt, sums_welcome=None,
                           spare_stream=Tensor(1 << 21, (1, H), F32), gemm_workspace=Tensor(WORKSPACE, (1 << 20,), F32))


def after(ffn, nxt):
    """What the block hands on."""
    ctx = context(nxt)
    return block(ffn).forward(ctx, Tensor(1 << 22, (1, H), F32), None, x_in=ctx.alloc((1, H)), next_norm=norm(), x_out=Tensor(1 << 23, (1, H), BF16))


def in_workspace(ctx, x):
    return Tensor(WORKSPACE, (3, 1, H), F32, layout="parts")


def in_the_steps_memory(ctx, x):
    t = ctx.alloc((1, 1, H), F32)
    return Tensor(t.ptr, t.shape, F32, layout="parts")


def test_partial_sums_of_a_product_wait_for_the_next_block():
    assert isinstance(after(in_workspace, block(in_workspace)), PendingNorm)


@pytest.mark.parametrize("ffn", [in_the_steps_memory, lambda ctx, x: ctx.alloc((1, H))])
def test_the_steps_own_memory_does_not_wait(ffn):
    """A routed layer's plane lies where the next block begins to allocate: its q | k | v row would be written over it by the product that reads it."""
    assert not isinstance(after(ffn, block(in_workspace)), PendingNorm)


def test_no_norm_waits_for_a_block_of_its_own_kind():
    class Own(Block):
        def forward(self, ctx, h, cache, **kw):
            raise AssertionError

    own = Own.__new__(Own)
    own.__dict__.update(block(in_workspace).__dict__)
    assert not isinstance(after(in_workspace, own), PendingNorm)
    assert not isinstance(after(in_workspace, None), PendingNorm)


@pytest.mark.parametrize("off,waits", [(0, True), (8, False), (16, True)])
def test_rows_that_16_byte_loads_do_not_reach(off, waits):
    """The products that make their own norm read 16 bytes at a time; a mixer's row elsewhere goes through the norm's kernel."""
    seen = []
    b = block(lambda ctx, x: (seen.append(x), ctx.alloc((1, H)))[1])
    b.ffn.takes_pending_norm = lambda ctx, size, planes: True
    b.mixer.forward = lambda ctx, x, cache: Tensor(8192 + off, (1, H), BF16)
    ctx = context(None)
    b.forward(ctx, Tensor(1 << 22, (1, H), F32), None, x_in=ctx.alloc((1, H)), next_norm=norm(), x_out=Tensor(1 << 23, (1, H), BF16))
    assert isinstance(seen[0], PendingNorm) == waits
