"""The key-split forward and dQ tilings against the default tilings on the same
inputs, fp32 outputs, at the edges of their 128-key steps, 32-key blocks and
64- and 128-row workgroups."""
import math

import pytest
import torch

from mimansm1_v1_amd import _lib
from mimansm1_v1_amd import attention as A

pytestmark = pytest.mark.gpu

# S = 1 .. 32: key groups without keys; 33 .. 64, 65 .. 127: groups whose block
# lies past the sequence, the step's second tile missing; 128, 129, 257: step edges
LENGTHS = [1, 31, 33, 64, 65, 97, 127, 128, 129, 193, 257, 400]
SPLIT = [i for i, c in enumerate(A.fwd_configs()) if c["schedule"] == "keysplit"]
SPLIT_DQ = [i for i, c in enumerate(A.tile_space("dq")) if c["schedule"] == "keysplit"]


def test_both_row_counts_are_compiled():
    assert len(SPLIT) == 2 and len(SPLIT_DQ) == 2


@pytest.mark.parametrize("H,Hkv,causal", [(10, 2, True), (10, 2, False), (8, 1, True), (3, 3, True), (3, 3, False)])
@pytest.mark.parametrize("S", LENGTHS)
def test_split_tilings_match_the_default(hip_device, S, H, Hkv, causal):
    lib, B, D = _lib.load(), 2, 128
    gen = torch.Generator(device=hip_device).manual_seed(S + H)
    rand = lambda n: torch.randn(B, S, n, D, device=hip_device, generator=gen).to(torch.bfloat16)
    q, k, v, do = rand(H), rand(Hkv), rand(Hkv), rand(H)
    shape = (B, S, H, Hkv, D, int(causal), D ** -0.5)
    sp = torch.cuda.current_stream(hip_device).cuda_stream

    def forward(tiles):
        o = torch.full((B, S, H, D), float("nan"), device=hip_device)
        lse = torch.full((B, H, S), float("nan"), device=hip_device)
        st = torch.zeros(lib.mm1_attn_fwd_state_size(*shape[:5]), dtype=torch.uint8, device=hip_device)
        assert lib.mm1_attn_fwd_f32(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr(),
                                    st.data_ptr(), st.numel(), *shape, tiles, sp) == 0
        return o, lse, st

    o0, lse0, st0 = forward(0)
    # each P is rounded to fp16 (2^-11) in the frame its tiling keeps, so O moves by
    # at most 2 x 2^-11 of the largest |V|; l and m are fp32 sums and maxima
    for tiles in SPLIT:
        o, lse, st = forward(tiles)
        assert (o - o0).abs().max() <= 2.0 ** -10 * v.abs().max().float()
        assert (lse - lse0).abs().max() <= 2.0 ** -18 * max(1.0, lse0.abs().max().item())
        nq = B * S * H * D * 2
        assert torch.equal(st[:nq], st0[:nq])                      # the fp16 Q for the backward

    ob = o0.to(torch.bfloat16)

    def backward(dq_tiles):
        dq = torch.full((B, S, H, D), float("nan"), device=hip_device)
        dk, dv = (torch.empty(B, S, Hkv, D, device=hip_device) for _ in range(2))
        ws = torch.empty(lib.mm1_attn_bwd_workspace_size(*shape[:5]), dtype=torch.uint8, device=hip_device)
        assert lib.mm1_attn_bwd_f32_tiles(ob.data_ptr(), do.data_ptr(), lse0.data_ptr(), st0.data_ptr(),
                                          st0.numel(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), ws.data_ptr(),
                                          ws.numel(), *shape, 0, dq_tiles, sp) == 0
        return dq, dk, dv

    # the same dS in every tiling: dQ differs by the order of an fp32 sum of S
    # terms dS K, 2 S 2^-24 sum |dS K| at most
    G = H // Hkv
    qd, kd, vd, dod, od = (t.double().transpose(1, 2) for t in (q, k, v, do, o0))
    kd, vd = (t.repeat_interleave(G, dim=1).contiguous() for t in (kd, vd))
    s = torch.matmul(qd, kd.transpose(-1, -2).contiguous()) / math.sqrt(D)
    if causal:
        s = s.masked_fill(torch.ones(S, S, dtype=torch.bool, device=hip_device).triu(1), -math.inf)
    ds = torch.softmax(s, -1) * (torch.matmul(dod, vd.transpose(-1, -2).contiguous())
                                 - (od * dod).sum(-1, keepdim=True)) / math.sqrt(D)
    size = torch.matmul(ds.abs(), kd.abs()).transpose(1, 2)
    dq0, dk0, dv0 = backward(0)
    for tiles in SPLIT_DQ:
        dq, dk, dv = backward(tiles)
        assert ((dq - dq0).abs().double() <= 2 * S * 2.0 ** -24 * 1.01 * size + 1e-7).all()
        assert torch.equal(dk, dk0) and torch.equal(dv, dv0)       # the partial sums in the dQ launch's tail
