"""Operations that several parts share; the one place where a kernel is chosen."""
from __future__ import annotations

import ctypes

from ..runtime.device import BF16, F32, Tensor

MEMORY_SIDE_CACHE = 256 << 20       # bytes

EPILOGUES = {None: 0, "softcap": 1, "gelu_tanh": 2, "silu": 3, "relu": 5, "clamped_swiglu": 6, "relu2": 7, "gelu": 8}
GATED = ("gelu_tanh", "silu", "relu", "clamped_swiglu")


def tuned_gemm(ctx, K: int) -> bool:
    """True when the matrix-core product serves this step (bf16, tuned kernels on,
    rows of K values that are whole 16-byte pieces)."""
    return ctx.dtype == BF16 and ctx.tuned and ctx.k.has("zk_gemm_bf16") and K % 8 == 0


def strip_flag(ctx, w: Tensor) -> int:
    """How a matrix-core product of few rows reads ``w``: 0 row by row, 1 in strips, 3 in strips and past the caches
    (``ctx.weights_read_once``: a step finds nothing there of what the last one read)."""
    if w.layout != "strip":
        return 0
    return 3 if getattr(ctx, "weights_read_once", False) else 1


def values_once(ctx, cache) -> int:
    """1 where decoded tokens' values of ``cache`` may be read past the caches: nothing reads them again before they have left those.
    That is so for a layer whose keys and values are its own, in a step that passes through more than the cache on the memory's side
    holds, by the weights alone or by what its requests have cached (an upper bound)."""
    if getattr(cache, "shared", False) or getattr(cache, "lent", False):
        return 0
    return int(getattr(ctx, "weights_read_once", False) or
               ctx.R * ctx.max_ctx * getattr(ctx, "cache_token_bytes", 0) > MEMORY_SIDE_CACHE)


class PendingNorm:
    """One row that is not made yet: next(h + post(sub)).  The product that reads it makes it itself and stores the
    new stream beside the old one, and a step of one token has a launch less between two products.  A block hands it only to a
    part whose ``takes_pending_norm(ctx, size, planes)`` says yes; the part launches one product with ``args`` and then calls ``done``.
    ``sub`` lies where nothing that runs before that product, nor the product itself, writes."""

    def __init__(self, ctx, sub: Tensor, post, h: Tensor, nxt):
        self.sub, self.post, self.h, self.nxt, self.spare = sub, post, h, nxt, ctx.spare_stream
        self.shape, self.dtype, self.layout = h.shape, ctx.dtype, "pending"

    @staticmethod
    def possible(ctx, h: Tensor, sub: Tensor) -> bool:
        return (h.shape[0] == 1 and ctx.dtype == BF16 and ctx.tuned and getattr(ctx, "spare_stream", None) is not None and
                ctx.k.has("zk_norm_gated_bf16") and (sub.layout == "parts" or (sub.layout == "rows" and sub.dtype == BF16)) and
                sub.ptr % 16 == 0 and h.ptr % 16 == 0)       # (the norm's own kernel takes rows from 8-byte addresses too)

    @staticmethod
    def outlasts_block(ctx, sub: Tensor) -> bool:
        """Whether ``sub`` may wait for the next block's first product: partial sums in the products' workspace, not what lies in the
        step's own memory, which that block hands out again (to the rows that the very product writes, while others of its blocks read)."""
        ws = getattr(ctx, "gemm_workspace", None)
        return sub.layout == "parts" and ws is not None and sub.ptr == ws.ptr

    def args(self):
        """The leading arguments of the products that take one."""
        post, nxt = self.post, self.nxt
        return (self.sub.ptr, self.sub.shape[0] if self.sub.layout == "parts" else 0, post.weight.ptr,
                float(post.spec.eps), int(post.spec.unit_offset), self.h.ptr,
                self.spare.ptr, nxt.weight.ptr, float(nxt.spec.eps), int(nxt.spec.unit_offset))

    def done(self) -> None:
        """The stream lies in the spare row from here on, and the old row is the spare one."""
        self.h.ptr, self.spare.ptr = self.spare.ptr, self.h.ptr
        self.h.owner, self.spare.owner = self.spare.owner, self.h.owner


def linear(ctx, x: Tensor, w: Tensor, out: Tensor, epilogue=None, cap: float = 0.0, last_of=None,
           sums_ok: bool = False, lda: int = 0, ldc: int = 0) -> Tensor:
    """out[M, N] = x[M, K] @ w[N, K]^T with float accumulation.

    ``out`` may be float32 (logits) or the activation type.  In the 32-bit
    library only the plain product exists; the bf16 library picks a matrix-core
    kernel by the number of rows.  ``epilogue`` (matrix-core product only):
    "softcap" applies cap * tanh(x / cap); "gelu_tanh" / "silu" / "relu" take w as
    [2N, K], gate rows first, and store act(gate) * up; "clamped_swiglu" likewise, with ``cap`` as
    its limit: g = min(gate, cap), u = clamp(up, -cap, cap), g sigmoid(1.702 g) (u + 1).

    "relu2" stores max(x, 0)^2, "gelu" x (1 + erf(x / sqrt(2))) / 2.  ``lda``: the distance between the rows of ``x`` in elements
    where they are the first K columns of wider rows (0: K).  ``ldc``: the same for the rows of ``out``, whose
    columns behind the N-th are left as they are (0: N; ``out`` is then [M, N], else [M, ldc]).

    ``last_of``: the part whose result this product is (it passes itself).  When the block
    that called that very part has said that partial sums are welcome (``ctx.sums_welcome`` is
    the part: the block's joining kernel adds them up itself) and the product splits K over
    blocks, the joining launch is left out: what comes back is a float32 tensor [P, M, N] with
    layout "parts" in the product's workspace instead of ``out``, to be read before the next
    product.  A part that another part calls is not the one the block named, so it never
    hands partial sums to a caller that does not expect them.  ``sums_ok``: the caller reads
    such a tensor itself, whoever called it.
    """
    M, K = x.shape
    gated = epilogue in GATED
    N, K2 = w.shape
    if gated:
        N //= 2
    if epilogue is not None and not tuned_gemm(ctx, K):
        raise ValueError("linear: epilogues belong to the matrix-core product")
    ldc = int(ldc) or N
    if ldc < N:
        raise ValueError(f"linear: rows {ldc} apart hold no {N} columns")
    if K != K2 or out.shape != (M, ldc):
        raise ValueError(f"linear: x {x.shape}, w {w.shape}, out {out.shape} do not fit")
    if x.dtype != ctx.dtype or w.dtype != ctx.dtype:
        raise ValueError(f"linear: operands must be {ctx.dtype}, got x {x.dtype}, w {w.dtype}")
    if out.dtype not in (F32, ctx.dtype):
        raise ValueError(f"linear: out must be float32 or {ctx.dtype}, got {out.dtype}")
    out_f32 = 1 if out.dtype == F32 else 0
    k = ctx.k
    strip = w.layout == "strip"
    lda = int(lda) or K
    if lda < K:
        raise ValueError(f"linear: rows {lda} apart hold no {K} columns")
    # the matrix-core product reads whole 16-byte pieces: rows that begin at such addresses
    tuned = tuned_gemm(ctx, K) and lda % 8 == 0 and x.ptr % 16 == 0
    if (strip or epilogue is not None) and not tuned:
        raise ValueError("linear: weights in strip layout and epilogues need the matrix-core product")
    if tuned:
        ws = getattr(ctx, "gemm_workspace", None)      # lets a product of few columns split K over blocks
        welcome = sums_ok or (last_of is not None and getattr(ctx, "sums_welcome", None) is last_of)
        parts = ctypes.c_int(0) if (welcome and ws is not None) else None
        k.zk_gemm_bf16(x.ptr, lda, w.ptr, out.ptr, ldc, out_f32, M, N, K, EPILOGUES[epilogue], float(cap),
                       strip_flag(ctx, w), ws.ptr if ws is not None else None,
                       ws.nbytes if ws is not None else 0, ctypes.byref(parts) if parts is not None else None,
                       ctx.stream)
        if parts is not None and parts.value > 0:
            return Tensor(ws.ptr, (parts.value, M, N), F32, ws.owner, layout="parts")
    else:
        k.zk_gemm_plain(x.ptr, lda, w.ptr, out.ptr, ldc, out_f32, M, N, K, ctx.stream)
    return out
