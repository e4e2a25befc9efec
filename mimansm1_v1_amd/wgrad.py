"""Weight gradients dW = A^T B of the bf16 projections around the attention
and the SwiGLU feed-forward, over all tokens.

A GEMM whose reduction runs over the B*S tokens (16,384 at the training
shapes) but whose output is only a weight's size (1792 x 1280 for wq|wk|wv,
3328 x 1280 for w_down) has too few output tiles to fill 256 CUs.  The package's
GEMM core splits its leftover tiles along the tokens over all CUs and adds the
fp32 partial sums in a fixed order (gemm.py: 1792 x 1280 x 16384 157 -> 101 us).
Where it does not apply, splitting the tokens into chunks gives hipBLASLt a
batched GEMM with `chunks` times the tiles; the chunks' products come out in
fp32 and are summed in fp32.  Either way the result is the same sum as one
GEMM, rounded once at the end; hipBLASLt's own GEMM runs on any other shape.
"""
from __future__ import annotations

import torch

from . import gemm


def wgrad(a: torch.Tensor, b: torch.Tensor, chunks: int, out_dtype=torch.float32) -> torch.Tensor:
    """sum over tokens t of a[t]^T b[t], accumulated in fp32 and rounded once
    to `out_dtype`: a [T, M], b [T, N] -> [M, N].  Without the GEMM core splits
    T into `chunks` when it divides evenly into chunks of at least 64 tokens;
    else one GEMM with fp32 output."""
    t, m = a.shape
    n = b.shape[1]
    if gemm.applies(a.t(), b.t()):
        return gemm.product(a.t(), b.t(), out_dtype=out_dtype)
    if chunks > 1 and t % chunks == 0 and t >= 64 * chunks:
        return torch.bmm(a.reshape(chunks, t // chunks, m).transpose(1, 2),
                         b.reshape(chunks, t // chunks, n).contiguous(),
                         out_dtype=torch.float32).sum(0).to(out_dtype)
    return torch.mm(a.t(), b, out_dtype=torch.float32).to(out_dtype)
