"""SwiGLU HIP kernels vs the oracle on identical seeded bf16 inputs (GPU only).

Kernel-level checks compare against the oracle's restatement of each
reference kernel on the same bf16 operands: the gate/up GEMM outputs are the
fp32 products rounded once, so the kernel (different fp32 summation order)
may differ from the oracle by at most one bf16 ulp; the gradient kernel is
elementwise on identical inputs (one ulp allowed for the exp2-based sigmoid).
The fused op is checked against the fp32 reference math with the reference
harness's own gate, max|d| / max|ref| < 3e-2 (swiglu_tilelang.py:551-555),
plus relative L2 <= 1e-2."""
from __future__ import annotations

import sys

import pytest
import torch
import torch.nn.functional as F

from oracle import swiglu as SW

pytestmark = pytest.mark.gpu

ULP_FRAC = 2.0 ** -7      # bf16 spacing relative to the leading power of two


def log(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def ulp(x: torch.Tensor) -> torch.Tensor:
    e = torch.floor(torch.log2(x.abs().clamp(min=2.0 ** -126)))
    return torch.pow(2.0, e) * ULP_FRAC


def assert_within_ulp(name, got, want, n_ulp=1.0, atol_rel=2e-6):
    """|got - want| <= n_ulp bf16 ulps of want, plus atol_rel * max|want| for
    values so close to zero that the fp32 summation error of a length-d dot
    product exceeds their ulp."""
    g, w = got.detach().double().cpu(), want.detach().double().cpu()
    err = (g - w).abs()
    bad = err > n_ulp * ulp(w) + atol_rel * w.abs().max()
    log(f"    {name}: max_abs {err.max().item():.3e}  beyond {n_ulp:g} ulp: {int(bad.sum())} of {w.numel()}")
    assert torch.isfinite(g).all(), name
    assert not bad.any(), f"{name}: {int(bad.sum())} elements beyond {n_ulp} ulp"


SHAPES = [(256, 1280, 3328), (300, 256, 256), (1, 128, 128), (129, 384, 128), (777, 1280, 384)]


@pytest.mark.parametrize("T,d,Fh", SHAPES, ids=[f"T{t}d{d}F{f}" for t, d, f in SHAPES])
def test_gate_up_modes_vs_oracle(hip_device, T, d, Fh):
    from mimansm1_v1_amd import swiglu as S
    log(f"[case] gate_up T={T} d={d} F={Fh}")
    x, wg, wu, _, _ = SW.make_inputs(T, d_model=d, ffn=Fh, seed=T + d, std=0.05)
    xd, gd, ud = (t.to(hip_device) for t in (x, wg, wu))
    gate, up = S.get_kernel("split", T, d, Fh)(xd, gd, ud)
    act = S.get_kernel("gate_up", T, d, Fh)(xd, gd, ud)
    g2, u2, act2 = S.get_kernel("train", T, d, Fh)(xd, gd, ud)
    torch.cuda.synchronize()
    want_g, want_u = SW.split(x, wg, wu)
    # the oracle rounds the fp32 products; compare both against the fp64 product
    g64, u64 = x.double() @ wg.double(), x.double() @ wu.double()
    assert_within_ulp("gate", gate, g64)
    assert_within_ulp("up", up, u64)
    assert_within_ulp("act (fp32 epilogue)", act, g64 * torch.sigmoid(g64) * u64, n_ulp=2.0)
    assert torch.equal(g2.cpu(), gate.cpu()) and torch.equal(u2.cpu(), up.cpu())
    # the kernel's exp2-based sigmoid and torch's may round one bf16 step apart
    assert_within_ulp("act (training rounding)", act2, SW.act_train(gate.cpu(), up.cpu()), n_ulp=2.0)
    # against the oracle's own rounding of the fp32 products (one ulp apart at most)
    assert_within_ulp("gate vs oracle", gate, want_g.float())
    assert_within_ulp("up vs oracle", up, want_u.float())


@pytest.mark.parametrize("T,Fh", [(256, 3328), (77, 64)])
def test_grad_kernel_vs_oracle(hip_device, T, Fh):
    from mimansm1_v1_amd import swiglu as S
    log(f"[case] grad T={T} F={Fh}")
    gen = torch.Generator().manual_seed(T)
    a, g, u = (torch.randn(T, Fh, generator=gen).mul(s).to(torch.bfloat16) for s in (1.0, 3.0, 2.0))
    ad, gd, ud = (t.to(hip_device) for t in (a, g, u))
    kern = S.get_kernel("grad", T, Fh)
    dg, du = kern(ad, gd, ud)
    buf = torch.empty(T, 2 * Fh, dtype=torch.bfloat16, device=hip_device)
    dg2, du2 = kern(ad, gd, ud, out=buf)
    torch.cuda.synchronize()
    wg, wu = SW.grad(a, g, u)
    assert_within_ulp("d_gate", dg, wg.float(), n_ulp=2.0)
    assert_within_ulp("d_up", du, wu.float(), n_ulp=2.0)
    assert torch.equal(dg2.cpu(), dg.cpu()) and torch.equal(du2.cpu(), du.cpu())
    assert torch.equal(buf[:, :Fh].cpu(), dg.cpu())


def _rel(got, want):
    g, w = got.detach().float().cpu(), want.detach().float().cpu()
    return ((g - w).abs().max() / w.abs().max().clamp(min=1e-6)).item(), ((g - w).norm() / w.norm()).item()


@pytest.mark.parametrize("T", [512, 4096])
def test_fused_swiglu_vs_fp32_reference(hip_device, T):
    """fused_swiglu forward and backward against autograd of the fp32
    reference math (the reference's check_gpu, swiglu_tilelang.py:497-556)."""
    from mimansm1_v1_amd import swiglu as S
    log(f"[case] fused_swiglu T={T} d=1280 F=3328")
    x, wg, wu, wd, go = SW.make_inputs(T, seed=T)
    leaves = [t.to(hip_device).requires_grad_(True) for t in (x, wg, wu, wd)]
    out = S.fused_swiglu(*leaves)
    out.backward(go.to(hip_device))
    got = [out] + [t.grad for t in leaves]
    want = SW.grads(*(t.to(hip_device) for t in (x, wg, wu, wd, go)))
    for name, a, b in zip(("out", "d_x", "d_w_gate", "d_w_up", "d_w_down"), got, want):
        rel, l2 = _rel(a, b)
        log(f"    {name:9s} max|d|/max|ref| {rel:.3e}  rel_l2 {l2:.3e}")
        assert rel < 3e-2 and l2 < 1e-2, name


def test_swiglu_module_hip_matches_math_backend(hip_device):
    from mimansm1_v1_amd import swiglu as S
    log("[case] SwiGLU module hip vs math")
    torch.manual_seed(0)
    ffn = S.SwiGLU(S.FFNConfig()).to(hip_device)
    x = torch.randn(2, 300, 1280, device=hip_device)
    y_hip = ffn(x, backend="hip")
    y_alias = ffn(x, backend="tilelang")
    y_math = ffn(x, backend="math")
    rel, l2 = _rel(y_hip, y_math)
    log(f"    out max|d|/max|ref| {rel:.3e}  rel_l2 {l2:.3e}")
    assert rel < 3e-2 and l2 < 1e-2
    assert torch.equal(y_hip, y_alias)
    xg = x.clone().requires_grad_(True)
    ffn(xg, backend="hip").sum().backward()
    grads_hip = [xg.grad] + [p.grad.clone() for p in ffn.parameters()]
    ffn.zero_grad()
    xm = x.clone().requires_grad_(True)
    ffn(xm, backend="math").sum().backward()
    grads_math = [xm.grad] + [p.grad for p in ffn.parameters()]
    for name, a, b in zip(("d_x", "d_w_gate", "d_w_up", "d_w_down"), grads_hip, grads_math):
        rel, l2 = _rel(a, b)
        log(f"    {name:9s} max|d|/max|ref| {rel:.3e}  rel_l2 {l2:.3e}")
        assert rel < 3e-2 and l2 < 1e-2, name


def test_swiglu_deterministic(hip_device):
    from mimansm1_v1_amd import swiglu as S
    log("[case] swiglu determinism")
    x, wg, wu, wd, go = (t.to(hip_device) for t in SW.make_inputs(1000, seed=5))
    runs = []
    for _ in range(2):
        leaves = [t.clone().requires_grad_(True) for t in (x, wg, wu, wd)]
        S.fused_swiglu(*leaves).backward(go)
        runs.append([t.grad.cpu() for t in leaves])
    for a, b in zip(*runs):
        assert torch.equal(a, b)


@pytest.mark.parametrize("T", [1, 31, 32, 33, 63, 64, 65, 127, 128, 129, 256, 320, 333])
@pytest.mark.parametrize("d,Fh", [(128, 128), (256, 640), (1280, 3328)])
def test_few_tokens_and_the_act_alone(hip_device, T, d, Fh):
    """The small tiles at the edges of their 64 tokens and 32 columns, on either
    side of the switch to the large ones: gate and up within half a bf16 ulp of
    the exact products plus fp32 rounding of the sums, the training mode's
    three outputs bitwise those of split mode and of the act-only call."""
    from mimansm1_v1_amd import swiglu as S
    gen = torch.Generator(device=hip_device).manual_seed(T)
    x = torch.randn(T, d, device=hip_device, generator=gen).to(torch.bfloat16)
    wg, wu = ((torch.randn(d, Fh, device=hip_device, generator=gen) * 0.05).to(torch.bfloat16) for _ in range(2))
    gate, up, act = S.get_kernel("train", T, d, Fh)(x, wg, wu)
    for got, w in ((gate, wg), (up, wu)):
        exact, size = x.double() @ w.double(), x.double().abs() @ w.double().abs()
        assert ((got.double() - exact).abs() <= 2.0 ** -8 * exact.abs() + d * 2.0 ** -24 * size).all()
    assert all(torch.equal(a, b) for a, b in zip((gate, up), S.get_kernel("split", T, d, Fh)(x, wg, wu)))
    assert torch.equal(act, S.get_kernel("train", T, d, Fh).act_only(x, wg, wu))
    w_down = wg.t().contiguous()
    out = S.fused_swiglu(x, wg, wu, w_down)                       # nothing needs a gradient
    kept = S.fused_swiglu(x.requires_grad_(True), wg, wu, w_down)
    with torch.no_grad():
        assert torch.equal(out, S.fused_swiglu(x, wg, wu, w_down))
    assert torch.equal(out, kept.detach()) and kept.requires_grad and not out.requires_grad


@pytest.mark.parametrize("kind,outputs,T", [("train", 3, 10244), ("split", 2, 15364), ("gate_up", 1, 30724), ("act", 1, 30724)])
def test_outputs_past_the_caches(hip_device, kind, outputs, T):
    """Outputs above 192 MiB leave with non-temporal stores: bitwise those of two
    halves of the tokens, which are below it."""
    from mimansm1_v1_amd import swiglu as S
    d, Fh, cut = 128, 3328, T // 512 * 256
    assert outputs * T * Fh * 2 > 192 << 20 > outputs * (T - cut) * Fh * 2
    gen = torch.Generator(device=hip_device).manual_seed(T)
    x = torch.randn(T, d, device=hip_device, generator=gen).to(torch.bfloat16)
    wg, wu = ((torch.randn(d, Fh, device=hip_device, generator=gen) * 0.05).to(torch.bfloat16) for _ in range(2))

    def run(rows):
        if kind == "act":
            return (S.get_kernel("train", rows.shape[0], d, Fh).act_only(rows, wg, wu),)
        out = S.get_kernel(kind, rows.shape[0], d, Fh)(rows, wg, wu)
        return out if isinstance(out, tuple) else (out,)

    whole, lo, hi = run(x), run(x[:cut]), run(x[cut:])
    assert len(whole) == outputs
    for a, b, c in zip(whole, lo, hi):
        assert torch.equal(a, torch.cat((b, c)))


def test_backward_on_the_core(hip_device, monkeypatch):
    """At 14,848 tokens every product of the backward but d_act, the joined d_x
    among them, runs on the GEMM core: the gradients are those of torch's products
    up to the bf16 roundings on the way (d_x: one against two)."""
    from mimansm1_v1_amd import gemm, swiglu as S
    T, d, Fh = 14848, 1280, 1280
    gen = torch.Generator(device=hip_device).manual_seed(1)
    rand = lambda *shape, std=1.0: (torch.randn(*shape, device=hip_device, generator=gen) * std).to(torch.bfloat16)
    leaves = [t.requires_grad_(True) for t in (rand(T, d), rand(d, Fh, std=0.03), rand(d, Fh, std=0.03), rand(Fh, d, std=0.03))]
    dy, taken = rand(T, d), []
    for name in ("applies", "applies_joined"):
        real = getattr(gemm, name)
        monkeypatch.setattr(gemm, name, lambda *a, real=real, name=name: (taken.append((name, real(*a))), taken[-1][1])[1])
    got = torch.autograd.grad(S.fused_swiglu(*leaves), leaves, dy)
    assert taken.count(("applies_joined", True)) == 1 and taken.count(("applies", True)) >= 3
    for name in ("applies", "applies_joined"):
        monkeypatch.setattr(gemm, name, lambda *a: False)
    for a, b in zip(got, torch.autograd.grad(S.fused_swiglu(*leaves), leaves, dy)):
        assert (a.double() - b.double()).norm() <= 2.0 ** -7 * b.double().norm()
