"""The plain bf16 products (mimansm1_v1_amd/gemm.py) against fp64 products of
the same operands: every layout, ragged edges of the tiles, both tile widths,
the split along K, joined weights, halved outputs and fp32 outputs."""
import pytest
import torch

from mimansm1_v1_amd import _lib, gemm

pytestmark = pytest.mark.gpu


def operand(rows, k, col, gen, dev, pad=0):
    """[rows, K], stored with K contiguous or (col) outermost, row stride padded."""
    inner, outer = (rows, k) if col else (k, rows)
    t = torch.randn(outer, inner + pad, device=dev, generator=gen).to(torch.bfloat16)[:, :inner]
    return t.t() if col else t


def check(out, x, w):
    """Within the rounding of the output plus that of fp32 sums over K: |err| <=
    u |exact| + K 2^-24 sum_k |x w|, u = 2^-8 (bf16, one ulp) or 0."""
    xd, wd = x.double().contiguous(), w.double().contiguous()
    exact = xd @ wd.t().contiguous()
    size = xd.abs() @ wd.abs().t().contiguous()
    u = 2.0 ** -8 if out.dtype == torch.bfloat16 else 0.0
    over = ((out.double() - exact).abs() - u * exact.abs() - x.shape[1] * 2.0 ** -24 * size).max().item()
    assert over <= 0, over


# (M, N, K), small tiles and large: smallest; ragged rows and columns of a tile; several tiles; a
# 320-column width; few tiles over a long K (split over all CUs, runs of one
# and of two tiles); fewer window pairs than CUs (empty runs); 257 tiles (one left over)
SHAPES = [(8, 8, 128), (256, 256, 128), (264, 520, 256), (776, 1288, 384), (1000, 320, 640),
          (512, 1280, 8192), (264, 264, 16384), (8, 8, 16384), (1280, 640, 6144), (65792, 256, 256),
          (64, 64, 128), (65, 72, 128), (128, 1792, 1280), (77, 1280, 3328), (1, 1280, 6656), (320, 1280, 1280),
          (5000, 1288, 640), (3000, 3336, 384), (4104, 328, 896), (1288, 1288, 16384)]


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_products_vs_fp64(hip_device, M, N, K, layout):
    gen = torch.Generator(device=hip_device).manual_seed(M + N + K)
    M = (M + 7) // 8 * 8 if layout == "tn" else M      # k-major operands: rows of 8
    x = operand(M, K, layout == "tn", gen, hip_device)
    w = operand(N, K, layout != "nt", gen, hip_device)
    for dtype in (torch.bfloat16, torch.float32):
        out = gemm.product(x, w, out_dtype=dtype)
        check(out, x, w)
        assert torch.equal(out, gemm.product(x, w, out_dtype=dtype))


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
def test_plan_that_depends_on_the_layout(hip_device, layout):
    """112 tiles: whole ones with x k-contiguous, split along k with both k-major."""
    gen = torch.Generator(device=hip_device).manual_seed(5)
    x, w = operand(3584, 4096, layout == "tn", gen, hip_device), operand(2048, 4096, layout != "nt", gen, hip_device)
    for dtype in (torch.bfloat16, torch.float32):
        check(gemm.product(x, w, out_dtype=dtype), x, w)


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("M,N,K,dtype", [(62608, 1608, 128, torch.bfloat16), (78648, 1280, 128, torch.bfloat16),
                                         (33352, 1608, 128, torch.float32), (31304, 1608, 128, torch.float32),
                                         (12088, 8328, 4096, torch.bfloat16), (32952, 3200, 4096, torch.bfloat16),
                                         (39328, 1280, 4096, torch.float32), (15736, 3200, 4096, torch.float32)])
def test_outputs_past_the_caches(hip_device, M, N, K, dtype, layout):
    """Above 192 MiB the output leaves with non-temporal stores: tiles of 256 and
    of 320 columns (in pairs), whole and, from the fifth on, split along k."""
    assert M * N * dtype.itemsize > 192 << 20
    assert (_lib.load().mm1_gemm_workspace_size(M, N, K, 0) > 0) == (K == 4096)
    gen = torch.Generator(device=hip_device).manual_seed(M + N)
    x, w = operand(M, K, layout == "tn", gen, hip_device), operand(N, K, layout != "nt", gen, hip_device)
    check(gemm.product(x, w, out_dtype=dtype), x, w)


@pytest.mark.parametrize("M", [1, 77, 255, 257, 333])
def test_ragged_rows_and_padded_strides(hip_device, M):
    gen = torch.Generator(device=hip_device).manual_seed(M)
    for col in (False, True):
        x = operand(M, 256, False, gen, hip_device, pad=8)
        w = operand(328, 256, col, gen, hip_device, pad=16)
        check(gemm.product(x, w), x, w)


@pytest.mark.parametrize("T,d,F", [(300, 640, 128), (4096, 1280, 3328), (2048, 256, 4160)])
def test_joined_weights_and_split_output(hip_device, T, d, F):
    gen = torch.Generator(device=hip_device).manual_seed(T)
    d_gu = operand(T, 2 * F, False, gen, hip_device)
    wg, wu = (operand(d, F, False, gen, hip_device) for _ in range(2))
    check(gemm.product(d_gu, wg, w1=wu), d_gu, torch.cat((wg, wu), dim=1))
    x = operand(d, T, True, gen, hip_device)
    lo, hi = gemm.product(x, d_gu.t(), split=F)
    check(lo, x, d_gu.t()[:F])
    check(hi, x, d_gu.t()[F:])


@pytest.mark.parametrize("K", [1, 7, 63, 64, 65, 127, 129, 1000, 4099, 16383])
def test_ragged_reduction_of_weight_gradients(hip_device, K):
    """Both operands k-major: the k rows past K, which memory may hold NaN at,
    count as zeros."""
    gen = torch.Generator(device=hip_device).manual_seed(K)
    for M, N in ((264, 1288), (1280, 640), (3080, 3336)):
        xs, ws = (torch.full((K + 130, n), float("nan"), dtype=torch.bfloat16, device=hip_device) for n in (M, N))
        for t in (xs, ws):
            t[:K] = torch.randn(K, t.shape[1], device=hip_device, generator=gen).to(torch.bfloat16)
        x, w = xs[:K].t(), ws[:K].t()
        for dtype in (torch.bfloat16, torch.float32):
            check(gemm.product(x, w, out_dtype=dtype), x, w)


def test_c_abi_refuses_what_the_kernels_do_not_take(hip_device):
    lib = _lib.load()
    t = torch.zeros(512 * 512, dtype=torch.bfloat16, device=hip_device)
    p = t.data_ptr()

    def call(x=p, lx=0, ldx=256, w=p, lw=0, ldw=256, w1=None, cut=0, out=p, out1=None, n_cut=0, ldo=256,
             M=64, N=64, K=256):
        return lib.mm1_gemm(x, lx, ldx, w, lw, ldw, w1, cut, out, out1, n_cut, ldo, 0, None, 0, M, N, K, None)

    assert call(x=None) == -1
    for bad in (dict(K=192), dict(N=60), dict(lx=1), dict(lx=2), dict(ldx=128), dict(ldw=252), dict(ldo=32),
                dict(cut=64), dict(w1=p, cut=32), dict(out1=p, n_cut=32), dict(M=0), dict(lx=1, lw=1, M=60),
                dict(M=1 << 29), dict(ldx=1 << 22)):
        assert call(**bad) == -2, bad
    assert call(x=p + 2) == -6
    need = lib.mm1_gemm_workspace_size(512, 1280, 8192, 0)
    assert need > 0
    big = torch.zeros(1280 * 8192, dtype=torch.bfloat16, device=hip_device).data_ptr()
    assert lib.mm1_gemm(big, 0, 8192, big, 0, 8192, None, 0, big, None, 0, 1280, 0, None, 0, 512, 1280, 8192,
                        None) == -4


@pytest.mark.parametrize("sizes", [(8, 0, 0, 0), (0, 24, 0, 8), (2048, 8, 2056, 0), (16, 1280 * 1280, 40, 1 << 20)])
def test_cast_of_several_tensors(hip_device, sizes):
    """One launch rounds the fp32 tensors to bf16 as torch does, specials
    included, one after the other."""
    src = [torch.randn(n, device=hip_device) * 3 for n in sizes]
    for t in src:
        if t.numel():
            t[:8] = torch.tensor([float("inf"), -float("inf"), float("nan"), 0.0, -0.0, 1e-40, 3.3895e38, 1.00390625])
    dst = torch.empty(sum(sizes), dtype=torch.bfloat16, device=hip_device)
    segments = [a for t in src for a in (t.data_ptr() if t.numel() else None, t.numel())]
    stream = torch.cuda.current_stream().cuda_stream
    lib = _lib.load()
    assert lib.mm1_cast_bf16(*segments, dst.data_ptr(), stream) == 0
    torch.testing.assert_close(dst, torch.cat(src).to(torch.bfloat16), rtol=0, atol=0, equal_nan=True)
    p = dst.data_ptr()
    for bad in ((None, 8), (p, 4), (p, -8), (p + 4, 8)):
        assert lib.mm1_cast_bf16(*bad, *segments[2:], dst.data_ptr(), stream) < 0, bad


def _second_derivatives(call, leaves, grad_out):
    """For each recorded first gradient of call(): None (no graph), the message
    of torch's refusal (mm with an out_dtype has no derivative), or the gradients
    of its sum of squares with respect to every leaf and grad_out."""
    first = torch.autograd.grad(call(), leaves, grad_out, create_graph=True)
    every, res = [*leaves, grad_out], []
    for g in first:
        try:
            res.append(torch.autograd.grad(g.float().square().sum(), every, retain_graph=True, allow_unused=True)
                       if g.requires_grad else None)
        except RuntimeError as exc:
            res.append(str(exc))
    return res


def _same_terms(got, want):
    assert [type(a) for a in got] == [type(b) for b in want]
    for a, b in zip(got, want):
        if not isinstance(b, tuple):
            assert a == b
            continue
        assert [p is None for p in a] == [q is None for q in b]
        for p, q in zip(a, b):
            assert q is None or (p.double() - q.double()).norm() <= 2.0 ** -6 * q.double().norm()


def _leaf(gen, *shape, std=1.0, dtype=torch.bfloat16):
    return (torch.randn(*shape, device=gen.device, generator=gen) * std).to(dtype).requires_grad_(True)


@pytest.mark.parametrize("which", ["linear", "swiglu"])
def test_recorded_backward_keeps_its_graph(hip_device, which, monkeypatch):
    """Under create_graph the backward's products are torch's at a size that the
    core takes too: the same terms of a second derivative, to rounding, as with
    torch's products alone.  (64 tokens: below the batched weight gradient.)"""
    from mimansm1_v1_amd import attention as A, swiglu as S
    gen = torch.Generator(device=hip_device).manual_seed(3)
    x, dy = _leaf(gen, 64, 1280), _leaf(gen, 64, 1280)
    if which == "linear":
        leaves = [x, _leaf(gen, 1280, 1280, std=0.02, dtype=torch.float32)]
        call = lambda: A.BF16Linear.apply(*leaves)
    else:
        leaves = [x, *(_leaf(gen, *s, std=0.02) for s in ((1280, 3328), (1280, 3328), (3328, 1280)))]
        call = lambda: S.fused_swiglu(*leaves)
    with torch.no_grad():
        assert gemm.applies(dy, _leaf(gen, 1280, 1280).t())
    got = _second_derivatives(call, leaves, dy)
    monkeypatch.setattr(gemm, "applies", lambda *a, **k: False)
    want = _second_derivatives(call, leaves, dy)
    assert any(isinstance(g, tuple) for g in want)
    _same_terms(got, want)


@pytest.mark.parametrize("T", [64, 4096])
def test_recorded_backward_of_the_head(hip_device, T, monkeypatch):
    """The same for the head, and for the tied head as through a transposed copy
    of its embedding."""
    from mimansm1_v1_amd import lm_head as L
    gen = torch.Generator(device=hip_device).manual_seed(T)
    h, emb = _leaf(gen, T, 1280, std=0.03), _leaf(gen, 8192, 1280, dtype=torch.float32)
    weight = emb.detach().t().bfloat16().contiguous().requires_grad_(True)
    gl = torch.ones((), device=hip_device, requires_grad=True)
    t = torch.randint(0, 8192, (T,), device=hip_device, generator=gen)
    got = _second_derivatives(lambda: L.fused_cross_entropy(h, weight, t), [h, weight], gl)
    tied = _second_derivatives(lambda: L.tied_cross_entropy(h, emb, t), [h, emb], gl)
    monkeypatch.setattr(gemm, "applies", lambda *a, **k: False)
    want = _second_derivatives(lambda: L.fused_cross_entropy(h, weight, t), [h, weight], gl)
    copied = _second_derivatives(
        lambda: L.fused_cross_entropy(h, emb.to(torch.bfloat16).t().contiguous(), t), [h, emb], gl)
    assert any(isinstance(g, tuple) for g in want)
    _same_terms(got, want)
    _same_terms(tied, copied)
    # without its copy the Function makes one: the same first gradients
    own = torch.autograd.grad(L.TiedCrossEntropy.apply(h, emb, t, 49152), [h, emb])
    for a, b in zip(own, torch.autograd.grad(L.tied_cross_entropy(h, emb, t), [h, emb])):
        assert torch.equal(a, b)
