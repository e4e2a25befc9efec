"""Plain bf16 products on the gfx950 GEMM core (csrc/gemm.hip): fp32
accumulation, one rounding, deterministic.

``product(x, w)`` is x w^T over the last axis of both 2-D operands, each given
as it lies in memory: a tensor whose reduction axis is contiguous, or a
transposed view of one whose reduction axis is outermost.  ``applies(x, w)``
says whether the kernels take (and are the faster choice for) the call; the
callers use torch's GEMM where it is False.
"""
from __future__ import annotations

import torch

from . import _lib

DTYPE = torch.bfloat16
ROW, COL = 0, 1                 # MM1_GEMM_ROW, MM1_GEMM_COL


def _layout(t):
    """(layout, row stride) of a 2-D operand [rows, K], or None."""
    if t.dim() != 2 or t.dtype != DTYPE or not t.is_cuda or t.data_ptr() % 16:
        return None
    rows, k = t.shape
    if t.stride(1) == 1 and t.stride(0) % 8 == 0 and t.stride(0) >= k:
        return ROW, t.stride(0)
    if t.stride(0) == 1 and t.stride(1) % 8 == 0 and t.stride(1) >= rows and rows % 8 == 0:
        return COL, t.stride(1)
    return None


def recorded(*tensors) -> bool:
    """Whether autograd records an operation on these (a backward under
    create_graph): the kernels' products leave no graph, torch's do."""
    return torch.is_grad_enabled() and any(t.requires_grad for t in tensors)


# Products that mm1_gemm_estimate_us puts at this or less run on its small tiles:
# torch's GEMM takes 21 us of host time a call, this 11 (two launches: 15).
SMALL_US = 14.0


def applies(x, w, small=True) -> bool:
    """Whether mm1_gemm takes x [M, K] w [N, K]^T (K a multiple of 128 unless
    both are k-major, N of 8, not x k-major with w k-contiguous) and was measured faster than
    hipBLASLt's GEMM at such a size (MI355X; T tokens, widths 1280 to 49152):

    From M N K = 2.4e10 on:
    * with w k-major: x k-major (weight gradients)
      1280 x 6656 x 16384 409 -> 309 us, 3328 x 1280 269 -> 174, 1280 x 49152
      1985 -> 1669, 1280 x 1280 130 -> 84; x k-contiguous 16384 x 1280 x 3328
      161 -> 114 us, x 1792 91 -> 65;
    * both k-contiguous where 320-column tiles fill a round of the CUs
      (16384 x 1280 x 1280 63 -> 50 us, x 6656 225 -> 218, x 49152 1656 ->
      1558) or the reduction is long enough to split (1024 x 1280 x 49152
      331 -> 182 us); hipBLASLt is faster elsewhere (16384 x 3328 x 1280: 136
      against 143 us).
    Below, too few tiles or windows are left per CU (1792 x 1280 x 4096, both
    k-major: 45 against 48 us) until the product is so small that the host's
    work decides: those run on the small tiles (`small`, SMALL_US)."""
    m, k = x.shape
    n = w.shape[0]
    if not x.is_cuda or m < 1 or n < 1 or k < 1 or recorded(x, w):
        return False
    few = m * n * k < 24 * 10 ** 9
    if few and not (small and 0 <= _lib.load().mm1_gemm_estimate_us(m, n, k) <= SMALL_US):
        return False
    lx, lw = _layout(x), _layout(w)
    if lx is None or lw is None or (lx[0] == COL and lw[0] == ROW):
        return False
    if (k % 128 and lx[0] == ROW) or n % 8 or w.shape[1] != k or w.device != x.device:
        return False
    for (layout, ld), rows in ((lx, m), (lw, n)):
        if (256 * ld + k if layout == ROW else 64 * ld + rows) >= 1 << 30 or rows > 1 << 26:
            return False
    if few or lw[0] == COL:
        return True
    return (n % 320 == 0 and m * n >= 230 * 256 * 320) or (k >= 16384 and m * n >= 16 * 256 * 256)


def applies_joined(x, w, w1) -> bool:
    """applies() for product(x, w, w1): the joined width counts."""
    k = w.shape[1]
    if x.shape[0] * w.shape[0] * 2 * k < 24 * 10 ** 9:
        return False
    return (_layout(w) is not None and _layout(w) == _layout(w1) and w.shape == w1.shape and not recorded(w1)
            and k % 128 == 0 and x.shape[1] == 2 * k and applies(x[:, :k], w))


def product(x, w, w1=None, out_dtype=DTYPE, split=None):
    """x [M, K] times w [N, K] transposed -> [M, N] in bf16 or fp32.  With w1,
    [w | w1] joined along K.  With ``split`` (a multiple of 64), the result as
    two tensors, columns [0, split) and [split, N)."""
    (lx, ldx), (lw, ldw) = _layout(x), _layout(w)
    m, k = x.shape
    n = w.shape[0]
    k_cut = 0
    if w1 is not None:
        if _layout(w1) != (lw, ldw) or w1.shape[0] != n:
            raise ValueError("w1 must have w's layout, stride and rows")
        k_cut = w.shape[1]
    if k != w.shape[1] + (w1.shape[1] if w1 is not None else 0):
        raise ValueError(f"reduction lengths differ: x has {k}")
    out1 = None
    if split is None:
        out = torch.empty(m, n, dtype=out_dtype, device=x.device)
    else:
        if n != 2 * split:
            raise ValueError("split halves the columns")
        out, out1 = (torch.empty(m, split, dtype=out_dtype, device=x.device) for _ in range(2))
    lib = _lib.load()
    ws_bytes = lib.mm1_gemm_workspace_size(m, n, k, int(w1 is not None))
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=x.device) if ws_bytes else None
    ptr = lambda t: None if t is None else t.data_ptr()
    rc = lib.mm1_gemm(x.data_ptr(), lx, ldx, w.data_ptr(), lw, ldw, ptr(w1), k_cut, out.data_ptr(), ptr(out1),
                      split or 0, out.stride(0), int(out_dtype == torch.float32), ptr(ws), ws_bytes, m, n, k,
                      torch._C._cuda_getCurrentRawStream(x.device.index))
    _lib.check(rc, "mm1_gemm")
    return out if split is None else (out, out1)
