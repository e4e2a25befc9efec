"""Plain bf16 products on the gfx950 GEMM core (csrc/gemm.hip): fp32
accumulation, one rounding, deterministic.

``product(x, w)`` is x w^T over the last axis of both 2-D operands, each given
as it lies in memory: a tensor whose reduction axis is contiguous, or a
transposed view of one whose reduction axis is outermost.  ``applies(x, w)``
says whether the kernels take (and are the faster choice for) the call; the
callers use torch's GEMM where it is False.
"""
from __future__ import annotations

import functools

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

FEW = 24 * 10 ** 9              # M N K below which large tiles are too few or their walks too short
LONG_K = 16384                  # reductions worth splitting over the CUs left idle
CUS = 256

# The library's tiles with their rate against its 256 x 256 (k-contiguous x),
# fitted to where it overtakes the core
LIBRARY_TILES = ((256, 256, 1.0), (192, 256, 0.85), (256, 160, 0.85), (256, 128, 0.9), (192, 128, 0.8))


def _fill(m, n, bm, bn) -> float:
    """Share of the CUs' time that whole rounds of bm x bn tiles spend on m x n outputs."""
    tiles = -(-m // bm) * -(-n // bn)
    return m * n / (bm * bn * CUS * -(-tiles // CUS))


@functools.lru_cache(maxsize=1024)
def pays(m, n, k, x_layout, w_layout, joined=False) -> bool:
    """Whether the large tiles were measured faster than hipBLASLt's GEMM for
    [m, k] x [n, k]^T, k over all of a joined w (MI355X, 1700 products of widths
    512 to 49152 and 256 to 65536 tokens; us, hipBLASLt -> the core):

    From M N K = 2.4e10 on (below, too few tiles or windows are left per CU:
    1792 x 1280 x 4096, both k-major, 45 -> 48), by how the rounds of tiles fill
    the CUs, which decides both sides' rate:
    * both k-major (weight gradients): 1280 x 6656 x 16384 425 -> 310, 1792 x 1280
      112 -> 102, 1280 x 49152 1976 -> 1850; not where 160-column tiles of the
      library fill exactly one round and K is neither short nor very long
      (8192 x 1280 x 8192 fp32 165 -> 213, x 16384 444 -> 362 in bf16);
    * x k-contiguous, K of LONG_K or more: the core splits K where its tiles leave
      CUs idle, at about 0.78 of a full round's rate (1024 x 1280 x 49152 345 ->
      181, w k-major 414 -> 172); the library is faster where one of its tiles
      fills more than that (8192 x 1280 x 49152, 160 columns: 869 -> 1086; 9741,
      192 rows: 915 -> 1354);
    * else where the core's 320 columns fill the rounds a tenth better than any
      tile of the library (16384 x 1280 x 3328, w k-major, 143 -> 107; x 1280,
      both k-contiguous, 58 -> 48; joined x 6656 268 -> 217), or nearly fill them
      at a width that its 256 columns do not divide (16384 x 4480 x 2048 304 ->
      241); not 65536 x 1280 x 1280 (159 -> 192), 3562 x 2048 x 4352 (62 -> 97),
      5662 x 1280 x 3328 (49 -> 63).  Both k-contiguous at a shorter K from 0.89
      of a round on (13312 x 1280 x 8192 at 0.81: 235 -> 283)."""
    if m * n * k < FEW:
        return False
    if x_layout == COL:
        one_round = m * n == 256 * 160 * CUS and (m % 256 == n % 160 == 0 or m % 160 == n % 256 == 0)
        return not (one_round and 3900 <= k <= 12600)
    wide = _fill(m, n, 256, 320) if n % 320 == 0 else 0.0
    library = max(rate * _fill(m, n, bm, bn) for bm, bn, rate in LIBRARY_TILES)
    if k >= LONG_K and not joined:
        return max(wide, 0.78) >= library and (w_layout == COL or m * n >= 16 * 256 * 256)
    if n % 256 and wide >= 0.8:
        return True
    return wide >= 1.1 * library and (w_layout == COL or wide >= 0.89)


def _operands(x, w):
    """The layouts of x [M, K] and w [N, K] if mm1_gemm takes them, else None:
    K a multiple of 128 unless both are k-major (then at most 2^28), N of 8, not
    x k-major with w k-contiguous, offsets inside 32 bits."""
    lx, lw = _layout(x), _layout(w)
    if lx is None or lw is None or (lx[0] == COL and lw[0] == ROW):
        return None
    m, k = x.shape
    n = w.shape[0]
    if (k % 128 and lx[0] == ROW) or k > 1 << 28 or n % 8 or w.device != x.device:
        return None
    for (layout, ld), rows in ((lx, m), (lw, n)):
        if (256 * ld + k if layout == ROW else 64 * ld + rows) >= 1 << 30 or rows > 1 << 26:
            return None
    return lx[0], lw[0]


def applies(x, w, small=True) -> bool:
    """Whether mm1_gemm takes x [M, K] w [N, K]^T and is the faster choice: by
    pays() for the large tiles, and (`small`) on the small ones where the product
    is so small that the host's work decides (SMALL_US).  Never where autograd
    would record the product."""
    m, k = x.shape
    n = w.shape[0]
    if not x.is_cuda or m < 1 or n < 1 or k < 1 or w.shape[1] != k or recorded(x, w):
        return False
    few = m * n * k < FEW
    if few and not (small and 0 <= _lib.load().mm1_gemm_estimate_us(m, n, k) <= SMALL_US):
        return False
    layouts = _operands(x, w)
    return layouts is not None and (few or pays(m, n, k, *layouts))


def applies_joined(x, w, w1) -> bool:
    """applies() for product(x, w, w1), on the large tiles: pays() over the joined
    width."""
    m, k = x.shape
    n, half = w.shape
    if not x.is_cuda or m < 1 or w.shape != w1.shape or k != 2 * half or half % 128 or recorded(x, w, w1):
        return False
    layouts = _operands(x, w)
    return layouts is not None and _layout(w) == _layout(w1) and pays(m, n, k, *layouts, joined=True)


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
