"""What a program built on this package has the GPU do, as timed and checked cases.

Each case is one call (or one forward and backward) of a public entry point:
the attention op, the QK-norm + RoPE op, the attention sublayer, the SwiGLU
feed-forward and the cross-entropy head, from short prompts to the training
shapes, whole and ragged sizes, causal and full attention, one and several
query heads per KV head, forward only and with gradients.

Interface: ``listed()`` and ``draw(rng)`` give cases (dicts of plain values),
``prepare(case, seed)`` the inputs and handles of one, ``run(state)`` one pass
and its outputs, ``work(case)`` the bytes and operations it cannot do without,
``tolerance(case)`` what two correct implementations may differ by, and
``exact(case, seed)`` the outputs in 64-bit arithmetic by plain torch.
"""
from __future__ import annotations

import atexit
import math
import os
import shutil
import tempfile

# The attention op searches its tilings at the first call of a shape and keeps
# the winner in the machine's store; a store of this process's own keeps the
# choice from depending on what ran on the machine before.
if "MM1_TUNED_STORE" not in os.environ:
    _store = tempfile.mkdtemp(prefix="mm1_tiles_")
    os.environ["MM1_TUNED_STORE"] = os.path.join(_store, "tuned_tiles.json")
    atexit.register(shutil.rmtree, _store, ignore_errors=True)

import torch  # noqa: E402

from mimansm1_v1_amd import attention, lm_head, swiglu  # noqa: E402

BF16 = torch.bfloat16
HEAD_DIM = 128
D_MODEL, FFN, VOCAB = 1280, 3328, 49152
THETA = 10_000.0


def _attn(batch, seq, heads=10, kv_heads=2, causal=True, train=True):
    return dict(kind="attn", batch=batch, seq=seq, heads=heads, kv_heads=kv_heads, causal=causal, train=train)


def _rope(batch, seq, heads=10, kv_heads=2, norm=True):
    return dict(kind="rope", batch=batch, seq=seq, heads=heads, kv_heads=kv_heads, norm=norm)


def _sublayer(batch, seq, train=True):
    return dict(kind="sublayer", batch=batch, seq=seq, train=train)


def _swiglu(tokens, d_model=D_MODEL, ffn=FFN, train=True, module=False):
    return dict(kind="swiglu", tokens=tokens, d_model=d_model, ffn=ffn, train=train, module=module)


def _head(tokens, d_model=D_MODEL, vocab=VOCAB, train=True, module=False, chunk=VOCAB):
    return dict(kind="head", tokens=tokens, d_model=d_model, vocab=vocab, train=train, module=module, chunk=chunk)


def listed():
    return [
        # a short prompt scored once: the attention op's smallest forward, where launches count
        dict(_attn(1, 512, train=False), name="attn_fwd_b1_s512"),
        # a training step on documents of an odd length: partial tiles everywhere
        dict(_attn(3, 1365), name="attn_train_b3_s1365"),
        # the first training stage's attention
        dict(_attn(8, 2048), name="attn_train_b8_s2048"),
        # the long-context training stage's attention
        dict(_attn(2, 8192), name="attn_train_b2_s8192"),
        # full (not causal) attention with a KV head per query head, as an encoder has it
        dict(_attn(2, 1000, heads=8, kv_heads=8, causal=False), name="attn_full_b2_s1000_mha"),
        # the sublayer's normalisation and rotation of Q and K alone, long sequences
        dict(_rope(4, 4095), name="rope_train_b4_s4095"),
        # fine-tuning on single short samples: the whole attention sublayer under autocast
        dict(_sublayer(1, 300), name="sublayer_train_b1_s300"),
        # the sublayer at the long-context training shape
        dict(_sublayer(2, 8192), name="sublayer_train_b2_s8192"),
        # the feed-forward of a short prompt, no gradients
        dict(_swiglu(77, train=False), name="swiglu_fwd_t77"),
        # the feed-forward of a training micro step
        dict(_swiglu(16384), name="swiglu_train_t16384"),
        # loss and gradients of a thousand tokens through the module of a head tied to the embedding
        dict(_head(1000, module=True), name="head_tied_train_t1000"),
        # loss and gradients of a training micro step over the whole vocabulary
        dict(_head(16384), name="head_train_t16384"),
    ]


def _log_int(rng, lo, hi):
    """A whole number spread over the logarithm of lo..hi, hi included."""
    return min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))


def draw(rng):
    kind = rng.choice(("attn", "attn", "attn", "rope", "sublayer", "swiglu", "swiglu", "head", "head"))
    if kind in ("attn", "rope", "sublayer"):
        seq = _log_int(rng, 16, 8192)
        batch = rng.randint(1, max(1, min(16, 16384 // seq)))
        if kind == "sublayer":
            return _sublayer(batch, seq, train=rng.random() < 0.7)
        heads, kv_heads = rng.choice(((10, 2), (10, 2), (10, 2), (8, 8), (8, 4), (8, 1)))
        if kind == "rope":
            return _rope(batch, seq, heads, kv_heads, norm=rng.random() < 0.8)
        return _attn(batch, seq, heads, kv_heads, causal=rng.random() < 0.8, train=rng.random() < 0.65)
    d_model = rng.choice((1280, 1280, 1280, 512, 2048))
    if kind == "swiglu":
        ffn = FFN if d_model == D_MODEL else 128 * rng.randint(d_model // 64, 3 * d_model // 128)
        return _swiglu(_log_int(rng, 1, 16384), d_model, ffn, train=rng.random() < 0.6, module=rng.random() < 0.3)
    d_model = min(d_model, D_MODEL)
    vocab = rng.choice((VOCAB, VOCAB, 32000, 8192))
    train = rng.random() < 0.6
    chunk = rng.choice((VOCAB, VOCAB, VOCAB, 8192)) if train else VOCAB
    return _head(_log_int(rng, 1, 16384 if chunk == VOCAB else 8192), d_model, vocab, train,
                 module=rng.random() < 0.3, chunk=chunk)


# ---------------------------------------------------------------------------
# Inputs
class _Draws:
    """Seeded tensors on the GPU, in the order they are asked for."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, std=1.0, mean=0.0, dtype=BF16):
        t = torch.randn(*shape, device="cuda", generator=self.gen)
        return t.mul_(std).add_(mean).to(dtype)

    def targets(self, tokens, vocab):
        """Token ids, one in sixteen ignored (padding, masked prompts)."""
        ids = torch.randint(0, vocab, (tokens,), device="cuda", generator=self.gen)
        drop = torch.rand(tokens, device="cuda", generator=self.gen) < 1 / 16
        drop[0] = False
        return ids.masked_fill(drop, lm_head.IGNORE_INDEX)


def _inputs(case, seed):
    r, kind = _Draws(seed), case["kind"]
    t = {}
    if kind == "attn":
        B, S, H, Hkv = (case[n] for n in ("batch", "seq", "heads", "kv_heads"))
        t["q"], t["k"], t["v"] = r.normal(B, S, H, HEAD_DIM), r.normal(B, S, Hkv, HEAD_DIM), r.normal(B, S, Hkv, HEAD_DIM)
        t["d_out"] = r.normal(B, S, H, HEAD_DIM) if case["train"] else None
    elif kind == "rope":
        B, S, H, Hkv = (case[n] for n in ("batch", "seq", "heads", "kv_heads"))
        t["qkv"] = r.normal(B, S, (H + 2 * Hkv) * HEAD_DIM)
        for name in ("wq", "wk"):
            t[name] = r.normal(HEAD_DIM, std=0.1, mean=1.0, dtype=torch.float32) if case["norm"] else None
        t["dq"], t["dk"], t["dv"] = r.normal(B, S, H, HEAD_DIM), r.normal(B, S, Hkv, HEAD_DIM), r.normal(B, S, Hkv, HEAD_DIM)
    elif kind == "sublayer":
        B, S = case["batch"], case["seq"]
        t["x"] = r.normal(B, S, D_MODEL, dtype=torch.float32)
        for name, rows in (("wq", 1280), ("wk", 256), ("wv", 256), ("wo", 1280)):
            t[name] = r.normal(rows, D_MODEL, std=0.02, dtype=torch.float32)
        for name in ("q_norm", "k_norm"):
            t[name] = r.normal(HEAD_DIM, std=0.1, mean=1.0, dtype=torch.float32)
        t["d_out"] = r.normal(B, S, D_MODEL) if case["train"] else None
    elif kind == "swiglu":
        T, d, f = case["tokens"], case["d_model"], case["ffn"]
        dtype = torch.float32 if case["module"] else BF16
        t["x"] = r.normal(T, d, dtype=dtype)
        t["w_gate"], t["w_up"], t["w_down"] = (r.normal(*shape, std=0.02, dtype=dtype) for shape in ((d, f), (d, f), (f, d)))
        t["d_out"] = r.normal(T, d, dtype=dtype) if case["train"] else None
    else:
        T, d, V = case["tokens"], case["d_model"], case["vocab"]
        t["targets"] = r.targets(T, V)
        if case["module"]:      # scaled by 1/sqrt(d) in the head: logits of deviation about 2
            t["hidden"] = r.normal(T, d, dtype=torch.float32)
            t["embedding"] = r.normal(V, d, std=2.0, dtype=torch.float32)
        else:
            t["hidden"] = r.normal(T, d)
            t["weight"] = r.normal(d, V, std=0.06)
    return t


class _State:
    def __init__(self, case, inputs):
        self.case, self.t = case, inputs
        self.module = self.leaves = None

    def grads_of(self, *tensors):
        self.leaves = [x.requires_grad_(True) for x in tensors]


def prepare(case, seed):
    s = _State(dict(case), _inputs(case, seed))
    t, kind = s.t, case["kind"]
    if kind == "attn":
        shape = (case["batch"], case["heads"], case["seq"], HEAD_DIM, case["causal"], case["heads"] // case["kv_heads"])
        attention.get_kernel("fwd", *shape)
        if case["train"]:
            attention.get_kernel("bwd", *shape)
            s.grads_of(t["q"], t["k"], t["v"])
    elif kind == "rope":
        rope = attention.Rotary(HEAD_DIM, 8192, THETA).to("cuda")
        t["cos"], t["sin"] = rope.cos, rope.sin
        s.grads_of(*(x for x in (t["qkv"], t["wq"], t["wk"]) if x is not None))
    elif kind == "sublayer":
        cfg = attention.AttnConfig()
        s.module = attention.Attention(cfg, attention.Rotary(HEAD_DIM, cfg.max_seq_len, THETA)).to("cuda")
        with torch.no_grad():
            for name in ("wq", "wk", "wv", "wo", "q_norm", "k_norm"):
                getattr(s.module, name).weight.copy_(t[name])
        attention.warmup(case["batch"], case["seq"], cfg)
        if case["train"]:
            s.grads_of(t["x"], *(getattr(s.module, n).weight for n in ("wq", "wk", "wv", "wo", "q_norm", "k_norm")))
    elif kind == "swiglu":
        if case["module"]:
            s.module = swiglu.SwiGLU(swiglu.FFNConfig(d_model=case["d_model"], ffn_hidden=case["ffn"])).to("cuda")
            with torch.no_grad():
                for name in ("w_gate", "w_up", "w_down"):
                    getattr(s.module, name).copy_(t[name])
                    t[name] = getattr(s.module, name)
        if case["train"]:
            s.grads_of(t["x"], t["w_gate"], t["w_up"], t["w_down"])
    else:
        if case["module"]:
            emb = torch.nn.Embedding(case["vocab"], case["d_model"], device="cuda", _weight=t["embedding"])
            cfg = lm_head.HeadConfig(d_model=case["d_model"], vocab=case["vocab"], chunk=case["chunk"])
            s.module = lm_head.LMHead(cfg, emb)
            t["embedding"] = emb.weight
        if case["train"]:
            s.grads_of(t["hidden"], t["embedding"] if case["module"] else t["weight"])
    return s


# ---------------------------------------------------------------------------
# One pass
def run(s):
    with torch.set_grad_enabled(s.leaves is not None):
        return _PASS[s.case["kind"]](s, s.case, s.t)


def _run_attn(s, case, t):
    groups = case["heads"] // case["kv_heads"]
    if not case["train"]:
        out, lse = attention.flash_attention_with_lse(t["q"], t["k"], t["v"], case["causal"], groups)
        return dict(out=out, lse=lse)
    out = attention.flash_attention(t["q"], t["k"], t["v"], case["causal"], groups)
    dq, dk, dv = torch.autograd.grad(out, s.leaves, t["d_out"])
    return dict(out=out, dq=dq, dk=dk, dv=dv)


def _run_rope(s, case, t):
    q, k, v = attention.qknorm_rope(t["qkv"], t["wq"], t["wk"], t["cos"], t["sin"], case["heads"], case["kv_heads"])
    grads = torch.autograd.grad((q, k, v), s.leaves, (t["dq"], t["dk"], t["dv"]))
    return dict(q=q, k=k, v=v, **dict(zip(("d_qkv", "d_wq", "d_wk"), grads)))


def _run_sublayer(s, case, t):
    with torch.autocast("cuda", dtype=BF16):
        y = s.module(t["x"])
    if not case["train"]:
        return dict(y=y)
    grads = torch.autograd.grad(y, s.leaves, t["d_out"])
    return dict(y=y, **dict(zip(("d_x", "d_wq", "d_wk", "d_wv", "d_wo", "d_q_norm", "d_k_norm"), grads)))


def _run_swiglu(s, case, t):
    out = s.module(t["x"]) if case["module"] else swiglu.fused_swiglu(t["x"], t["w_gate"], t["w_up"], t["w_down"])
    if not case["train"]:
        return dict(out=out)
    grads = torch.autograd.grad(out, s.leaves, t["d_out"])
    return dict(out=out, **dict(zip(("d_x", "d_w_gate", "d_w_up", "d_w_down"), grads)))


def _run_head(s, case, t):
    if case["module"]:
        loss = s.module(t["hidden"], t["targets"])
    elif not case["train"]:     # scoring: every token's log-sum-exp, target logit and loss
        lse, target_logit, losses = lm_head.get_kernel((case["tokens"], case["d_model"], case["vocab"])).forward(
            t["hidden"], t["weight"], t["targets"])
        return dict(lse=lse, target_logit=target_logit, losses=losses)
    else:
        loss = lm_head.fused_cross_entropy(t["hidden"], t["weight"], t["targets"], case["chunk"])
    if not case["train"]:
        return dict(loss=loss)
    d_hidden, d_weight = torch.autograd.grad(loss, s.leaves)
    return dict(loss=loss, d_hidden=d_hidden, d_weight=d_weight)


_PASS = dict(attn=_run_attn, rope=_run_rope, sublayer=_run_sublayer, swiglu=_run_swiglu, head=_run_head)


# ---------------------------------------------------------------------------
# What a pass cannot do without
def work(case):
    kind, train = case["kind"], case.get("train", True)
    if kind == "attn":
        return _attn_work(case["batch"], case["seq"], case["heads"], case["kv_heads"], case["causal"], train)
    if kind == "rope":
        rows = case["batch"] * case["seq"] * (case["heads"] + 2 * case["kv_heads"]) * HEAD_DIM
        # qkv and the three gradients in; q, k, v and d_qkv out
        return dict(bytes=4 * 2 * rows, flops=0)
    if kind == "sublayer":
        tokens = case["batch"] * case["seq"]
        weights = D_MODEL * (1792 + 1280)
        w = _attn_work(case["batch"], case["seq"], 10, 2, True, train)
        flops = 2 * tokens * weights * (3 if train else 1) + w["flops"]
        # x (fp32), weights (fp32) in, y (bf16) out; the gradients of all three
        nbytes = tokens * D_MODEL * 6 + 4 * weights + (tokens * D_MODEL * 8 + 4 * weights if train else 0)
        return dict(bytes=nbytes, flops=flops)
    if kind == "swiglu":
        T, d, f = case["tokens"], case["d_model"], case["ffn"]
        elem = 4 if case["module"] else 2
        flops = 6 * T * d * f * (3 if train else 1)
        return dict(bytes=elem * (2 * T * d + 3 * d * f + (2 * T * d + 3 * d * f if train else 0)), flops=flops)
    T, d, V = case["tokens"], case["d_model"], case["vocab"]
    elem = 4 if case["module"] else 2
    flops = 2 * T * d * V * (3 if train else 1)
    return dict(bytes=elem * (T * d + d * V) * (2 if train else 1) + 8 * T, flops=flops)


def _attn_work(B, S, H, Hkv, causal, train):
    pairs = B * H * (S * (S + 1) // 2 if causal else S * S)
    rows = B * S * (2 * H + 2 * Hkv) * HEAD_DIM          # q, k, v in, out
    nbytes = 2 * rows + 4 * B * H * S
    if train:
        nbytes += 2 * rows                               # d_out in, dq, dk, dv out
    return dict(bytes=nbytes, flops=2 * HEAD_DIM * pairs * (7 if train else 2))


def tolerance(case):
    return dict(_TOLERANCE[case["kind"], case.get("train", True)])


# Each about four times the relative error that the outputs show against the
# 64-bit values: bf16 results of fp32 sums (attention, RoPE, head gradients),
# of chains of bf16 products (feed-forward, sublayer), and fp32 results of
# fp32 sums (the head's log-sum-exp and losses).
_TOLERANCE = {
    ("attn", False): {"rel": 7e-3},
    ("attn", True): {"rel": 7e-3},
    ("rope", True): {"rel": 1.2e-2},
    ("sublayer", False): {"rel": 2e-2},
    ("sublayer", True): {"rel": 2e-2},
    ("swiglu", False): {"rel": 2e-2},
    ("swiglu", True): {"rel": 2e-2},
    ("head", False): {"rel": 2e-5},
    ("head", True): {"rel": 1.4e-2},
}


# ---------------------------------------------------------------------------
# The same in 64 bits
def exact(case, seed):
    t = {n: None if x is None else x if x.dtype == torch.int64 else x.double() for n, x in _inputs(case, seed).items()}
    with torch.no_grad():
        return _EXACT[case["kind"]](case, t)


def _attention64(q, k, v, causal, d_out=None):
    """(out, lse in log2 units, dq, dk, dv) of softmax attention, one head at a time."""
    B, S, H, D = q.shape
    groups = H // k.shape[2]
    scale = 1.0 / math.sqrt(D)
    out, lse = torch.empty_like(q), q.new_empty(B, H, S)
    dq, dk, dv = torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v)
    for b in range(B):
        for h in range(H):
            g = h // groups
            qh, kh, vh = (x.contiguous() for x in (q[b, :, h], k[b, :, g], v[b, :, g]))
            s = (qh @ kh.t().contiguous()).mul_(scale)
            if causal:
                s.masked_fill_(torch.ones(S, S, dtype=torch.bool, device=s.device).triu_(1), -math.inf)
            l = torch.logsumexp(s, dim=1)
            p = s.sub_(l[:, None]).exp_()
            o = p @ vh
            out[b, :, h], lse[b, h] = o, l / math.log(2.0)
            if d_out is None:
                continue
            do = d_out[b, :, h].contiguous()
            dv[b, :, g] += p.t().contiguous() @ do
            ds = (do @ vh.t().contiguous()).sub_((o * do).sum(1, keepdim=True)).mul_(p).mul_(scale)
            dq[b, :, h] = ds @ kh
            dk[b, :, g] += ds.t().contiguous() @ qh
    return out, lse, dq, dk, dv


def _exact_attn(case, t):
    out, lse, dq, dk, dv = _attention64(t["q"], t["k"], t["v"], case["causal"], t["d_out"])
    return dict(out=out, dq=dq, dk=dk, dv=dv) if case["train"] else dict(out=out, lse=lse)


def _tables64(seq, device):
    freq = THETA ** (-torch.arange(0, HEAD_DIM, 2, dtype=torch.float64, device=device) / HEAD_DIM)
    angle = (torch.arange(seq, dtype=torch.float64, device=device)[:, None] * freq).repeat(1, 2)[:, None]
    return angle.cos(), angle.sin()


def _half(x, sign):
    lo, hi = x.chunk(2, dim=-1)
    return torch.cat((-sign * hi, sign * lo), dim=-1)


def _norm_rope64(x, w, eps=1e-5):
    """Rows x [B,S,n,D] normalised, weighted and rotated, and their pullback."""
    cos, sin = _tables64(x.shape[1], x.device)
    r = (x.square().mean(-1, keepdim=True) + eps).rsqrt() if w is not None else torch.ones_like(x[..., :1])
    y = x * r * (w if w is not None else 1.0)

    def back(dz):
        dy = dz * cos + _half(dz * sin, -1)
        if w is None:
            return dy, None
        wd = dy * w
        dx = r * wd - x * r ** 3 * (wd * x).mean(-1, keepdim=True)
        return dx, (dy * x * r).sum((0, 1, 2))

    return y * cos + _half(y, 1) * sin, back


def _split_heads(qkv, heads, kv_heads):
    x = qkv.unflatten(-1, (heads + 2 * kv_heads, HEAD_DIM))
    return x[:, :, :heads], x[:, :, heads:heads + kv_heads], x[:, :, heads + kv_heads:]


def _exact_rope(case, t):
    q, k, v = _split_heads(t["qkv"], case["heads"], case["kv_heads"])
    (qr, qb), (kr, kb) = _norm_rope64(q, t["wq"]), _norm_rope64(k, t["wk"])
    (dq, dwq), (dk, dwk) = qb(t["dq"]), kb(t["dk"])
    res = dict(q=qr, k=kr, v=v, d_qkv=torch.cat((dq, dk, t["dv"]), dim=2).flatten(2))
    if case["norm"]:
        res.update(d_wq=dwq, d_wk=dwk)
    return res


def _exact_sublayer(case, t):
    w = torch.cat((t["wq"], t["wk"], t["wv"]))
    x = t["x"]
    q, k, v = _split_heads(x @ w.t(), 10, 2)
    (qr, qb), (kr, kb) = _norm_rope64(q, t["q_norm"]), _norm_rope64(k, t["k_norm"])
    wo, d_y = t["wo"], t["d_out"]
    d_attn = None if d_y is None else (d_y @ wo).unflatten(-1, (10, HEAD_DIM))
    out, _, dq, dk, dv = _attention64(qr, kr, v, True, d_attn)
    y = out.flatten(2) @ wo.t()
    if d_y is None:
        return dict(y=y)
    (dq, d_qn), (dk, d_kn) = qb(dq), kb(dk)
    d_qkv = torch.cat((dq, dk, dv), dim=2).flatten(2)
    rows = lambda z: z.flatten(0, 1)  # noqa: E731
    d_w = rows(d_qkv).t() @ rows(x)
    return dict(y=y, d_x=d_qkv @ w, d_wq=d_w[:1280], d_wk=d_w[1280:1536], d_wv=d_w[1536:],
                d_wo=rows(d_y).t() @ rows(out.flatten(2)), d_q_norm=d_qn, d_k_norm=d_kn)


def _exact_swiglu(case, t):
    x, wg, wu, wd, dy = (t[n] for n in ("x", "w_gate", "w_up", "w_down", "d_out"))
    g, u = x @ wg, x @ wu
    s = torch.sigmoid(g)
    act = g * s * u
    out = act @ wd
    if dy is None:
        return dict(out=out)
    da = dy @ wd.t()
    dg, du = da * u * s * (1 + g * (1 - s)), da * g * s
    return dict(out=out, d_x=dg @ wg.t() + du @ wu.t(), d_w_gate=x.t() @ dg, d_w_up=x.t() @ du, d_w_down=act.t() @ dy)


def _exact_head(case, t):
    targets = t["targets"]
    scale = case["d_model"] ** -0.5 if case["module"] else 1.0
    h, w = t["hidden"] * scale, t["embedding"].t() if case["module"] else t["weight"]
    valid = targets != lm_head.IGNORE_INDEX
    at = targets.clamp(min=0)[:, None]
    logits = h @ w
    lse = torch.logsumexp(logits, dim=1)
    count = valid.sum()
    target_logit = logits.gather(1, at)[:, 0]
    losses = (lse - target_logit) * valid
    loss = losses.sum() / count
    if not case["train"] and not case["module"]:
        return dict(lse=lse, target_logit=target_logit, losses=losses)
    if not case["train"]:
        return dict(loss=loss)
    dl = logits.sub_(lse[:, None]).exp_()
    dl.scatter_add_(1, at, torch.full_like(at, -1.0, dtype=dl.dtype))
    dl.mul_((valid / count)[:, None])
    d_w = h.t() @ dl
    return dict(loss=loss, d_hidden=dl @ w.t() * scale, d_weight=d_w.t() if case["module"] else d_w)


_EXACT = dict(attn=_exact_attn, rope=_exact_rope, sublayer=_exact_sublayer, swiglu=_exact_swiglu, head=_exact_head)
