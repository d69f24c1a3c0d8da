"""Performance cases of the LoRA training step: what a user's program calls, over the
sizes it calls it with.

Families (every one through the public `llmt` binding):

  layer  one decoder layer of Qwen3-1.7B, forward and backward (Context.layer_forward /
         layer_backward): dx, the layer output and the eight adapter gradients
  head   the lm_head with the fused cross entropy and its dX over the 151,936-word
         vocabulary (Context.head_ce)
  block  the attention block, QK-norm + RoPE + causal GQA attention forward and backward
         (attention_block_bwd)
  attn   the attention operators on their own (attention_fwd, attention_bwd)
  step   the whole 28-layer training step as a driver runs it: one HIP graph a step,
         forward, cross entropy, backward and AdamW (Context.step)

`wfmt` is the frozen weights' format, "f16" or "i8" (int8 rows with fp16 scales).
"""
import math
import sys
from pathlib import Path

import torch
import torch.utils.checkpoint

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "llm.cu_amd"))
import llmt  # noqa: E402

H, NQ, NKV, HD, I, V, L, R = 2048, 16, 8, 128, 6144, 151936, 28, 16
Q, KV = NQ * HD, NKV * HD
EPS, THETA, SCALE = 1e-6, 1e6, 2.0
MATS = (("wq", Q, H), ("wk", KV, H), ("wv", KV, H), ("wo", H, Q), ("w_gate", I, H),
        ("w_up", I, H), ("w_down", H, I))
PROJ = (("wq", Q, H), ("wk", KV, H), ("wv", KV, H), ("wo", H, Q))
LAYER_PARAMS = sum(o * i for _, o, i in MATS)
LORA_LAYER = sum(R * (o + i) for _, o, i in PROJ)


def listed():
    return [
        # a prompt-sized sequence: launches and round trips are all there is
        dict(name="layer_f16_b1s32", kind="layer", wfmt="f16", B=1, S=32),
        # the headline step's layer (B1 x S128)
        dict(name="layer_f16_b1s128", kind="layer", wfmt="f16", B=1, S=128),
        # a few short documents of a length that is no power of two
        dict(name="layer_f16_b3s208", kind="layer", wfmt="f16", B=3, S=208),
        # the same layer on int8 frozen weights at the headline size
        dict(name="layer_i8_b1s128", kind="layer", wfmt="i8", B=1, S=128),
        # int8 fine-tuning in batches of an uneven length
        dict(name="layer_i8_b5s400", kind="layer", wfmt="i8", B=5, S=400),
        # the large-batch int8 configuration's layer (B8 x S512)
        dict(name="layer_i8_b8s512", kind="layer", wfmt="i8", B=8, S=512),
        # the loss and its gradient at the headline size, dlogits wanted
        dict(name="head_b1s128", kind="head", B=1, S=128, dlogits=True),
        # the loss of two uneven sequences, as a step takes it
        dict(name="head_b2s168", kind="head", B=2, S=168, dlogits=False),
        # the attention stress configuration: long sequences
        dict(name="block_b4s2048", kind="block", B=4, S=2048, nq=16, nkv=8),
        # attention of short documents of odd length, called as an operator
        dict(name="attn_b3s333", kind="attn", B=3, S=333, nq=16, nkv=8),
        # the headline step (B1 x S128, fp16 frozen weights)
        dict(name="step_f16_b1s128", kind="step", wfmt="f16", B=1, S=128),
        # the training driver's default sequence length and batch
        dict(name="step_f16_b1s512", kind="step", wfmt="f16", B=1, S=512),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "head", "block", "attn", "step"])
    if kind == "layer":  # batch * seq_len has to be a multiple of 16
        B = rng.choice([1, 1, 2, 3, 4, 5, 6, 8])
        unit = 16 // math.gcd(16, B)
        T = _log(rng, 24, 4096)
        S = max(unit, T // B // unit * unit)
        return dict(kind=kind, wfmt=rng.choice(["f16", "i8"]), B=B, S=S)
    if kind == "head":
        B = rng.choice([1, 1, 2, 3, 4])
        unit = 16 // math.gcd(16, B)
        S = max(unit, _log(rng, 16, 1024) // B // unit * unit)
        return dict(kind=kind, B=B, S=S, dlogits=rng.choice([True, False]))
    if kind in ("block", "attn"):
        nq, nkv = rng.choice([(16, 8), (16, 8), (8, 4), (32, 8), (8, 8)])
        S = _log(rng, 40, 4000)
        most = 4 * 16 * 2048 * 2048 // (nq * S * S)
        return dict(kind=kind, B=rng.randint(1, max(1, min(8, most))), S=S, nq=nq, nkv=nkv)
    B = rng.choice([1, 1, 2, 3])
    return dict(kind=kind, wfmt=rng.choice(["f16", "i8"]), B=B, S=max(9, _log(rng, 24, 510) // B))


# ---------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, shape, std=1.0, dtype=torch.float32):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).mul_(std).to(dtype)


def _quantize(w):
    """int8 rows with the reference's recipe (max|w| / 127, round half to even), fp16 scales."""
    s = w.abs().amax(1) / 127.0
    q = (w * (1.0 / s)[:, None]).clamp_(-127, 127).round_().to(torch.int8)
    return q, s.half()


def _layer_weights(g, wfmt):
    """The seven frozen matrices in the order of MATS (fp16, or pairs (q, scale)) and norms."""
    ws = [_randn(g, (o, i), 0.02, torch.float16) for _, o, i in MATS]
    if wfmt == "i8":
        ws = [_quantize(w.float()) for w in ws]
    norms = [1.0 + _randn(g, (n,), 0.1) for n in (H, H, HD, HD)]
    return ws, norms


def _adapters(g, layers):
    """A flat adapter arena: layer by layer, q, k, v, o, A then B."""
    parts = []
    for _ in range(layers):
        for _, o, i in PROJ:
            parts.append(_randn(g, (R * i,), 1.0 / math.sqrt(H)))
            parts.append(_randn(g, (o * R,), 0.01))
    return torch.cat(parts)


def _set_layer(ctx, l, ws, norms, wfmt):
    if wfmt == "i8":
        ctx.set_layer_i8(l, [w[0] for w in ws], [w[1] for w in ws], *norms)
    else:
        ctx.set_layer_f16(l, *ws, *norms)


def _dims(layers, vocab):
    d = llmt.qwen3_dims()
    d.n_layers, d.vocab = layers, vocab
    return d


def _inputs(case, g):
    """The call's own inputs (after the weights in the seed's order)."""
    B, S = case["B"], case["S"]
    if case["kind"] == "layer":
        return dict(x=_randn(g, (B * S, H)), dy=_randn(g, (B * S, H)))
    if case["kind"] == "head":
        x = _randn(g, (B * S, H), 1.0, torch.float16)
        tgt = torch.randint(0, V, (B, S), generator=g, device="cuda", dtype=torch.int32)
        return dict(x=x, tgt=tgt)
    if case["kind"] == "step":
        win = torch.randint(0, V, (B, S + 1), generator=g, device="cuda", dtype=torch.int32)
        return dict(tok=win[:, :-1].contiguous(), tgt=win[:, 1:].contiguous())
    nq, nkv = case["nq"], case["nkv"]
    f16 = torch.float16
    got = dict(q=_randn(g, (B, S, nq, HD), 1.0, f16), k=_randn(g, (B, S, nkv, HD), 1.0, f16),
               v=_randn(g, (B, S, nkv, HD), 1.0, f16))
    if case["kind"] == "block":
        got.update(do=_randn(g, (B, S, nq, HD), 1.0, f16), qn=1.0 + _randn(g, (HD,), 0.1),
                   kn=1.0 + _randn(g, (HD,), 0.1))
    else:
        got.update(do=_randn(g, (B, S, nq, HD)))
    return got


def prepare(case, seed):
    g = _gen(seed)
    kind, B, S = case["kind"], case["B"], case["S"]
    state = dict(case=case)
    if kind == "layer":
        ctx = llmt.Context(_dims(1, 256), B, S, int8=case["wfmt"] == "i8")
        _set_layer(ctx, 0, *_layer_weights(g, case["wfmt"]), case["wfmt"])
        ctx.lora_set("param", _adapters(g, 1))
        state["ctx"] = ctx
    elif kind == "head":
        ctx = llmt.Context(_dims(1, V), B, S)
        ctx.set_embed_f16(_randn(g, (V, H), 0.02, torch.float16), torch.ones(H, device="cuda"))
        state["ctx"] = ctx
    elif kind == "step":
        ctx = llmt.Context(_dims(L, V), B, S, int8=case["wfmt"] == "i8")
        for l in range(L):
            _set_layer(ctx, l, *_layer_weights(g, case["wfmt"]), case["wfmt"])
        ctx.set_embed_f16(_randn(g, (V, H), 0.02, torch.float16), 1.0 + _randn(g, (H,), 0.1))
        ctx.lora_set("param", _adapters(g, L))
        ctx.set_graph(True)
        state.update(ctx=ctx, n=0, hp=llmt.hparams())
    state.update(_inputs(case, g))
    return state


def run(s):
    case = s["case"]
    kind, B, S = case["kind"], case["B"], case["S"]
    if kind == "layer":
        ctx = s["ctx"]
        y = ctx.layer_forward(0, s["x"], B)
        dx = ctx.layer_backward(0, s["dy"], B)
        return dict(y=y, dx=dx, grads=ctx.lora_get("grad"))
    if kind == "head":
        loss, dlogits, dx = s["ctx"].head_ce(s["x"], s["tgt"], want_dlogits=case["dlogits"])
        return dict(loss=loss, dx=dx, dlogits=dlogits)
    if kind == "block":
        return llmt.attention_block_bwd(s["q"], s["k"], s["v"], s["qn"], s["kn"], s["do"],
                                        THETA, EPS)
    if kind == "attn":
        o, lse = llmt.attention_fwd(s["q"], s["k"], s["v"])
        return (o, lse) + llmt.attention_bwd(s["q"], s["k"], s["v"], o, lse, s["do"])
    s["n"] += 1
    ctx = s["ctx"]
    loss = ctx.step(s["tok"], s["tgt"], s["hp"], s["n"])
    return dict(loss=loss, logits=ctx.logits(B * S), grads=ctx.lora_get("grad"))


# ---------------------------------------------------------------- cost and accuracy

def _causal(B, S, nq, products):
    """flops of `products` causal S x S x 128 products of every query head."""
    return products * 2.0 * B * nq * (S * (S + 1) / 2) * HD


def work(case):
    kind, B, S = case["kind"], case["B"], case["S"]
    T = B * S
    wb = 1 if case.get("wfmt") == "i8" else 2
    # per layer: the weights once forward and once backward, forward and dX
    # products, the LoRA terms, two forward and five backward attention products
    lay_b = 2.0 * LAYER_PARAMS * wb + 2 * 4.0 * LORA_LAYER
    lay_f = 4.0 * T * LAYER_PARAMS + 6.0 * T * LORA_LAYER + _causal(B, S, NQ, 7)
    if kind == "layer":
        return dict(bytes=lay_b + 4 * 4.0 * T * H, flops=lay_f)
    # the head: its matrix once for the logits and once for dX
    head_b = 2 * 2.0 * V * H + T * H * (2 + 4.0) + (4.0 * T * V if case.get("dlogits") else 0)
    head_f = 4.0 * T * V * H
    if kind == "head":
        return dict(bytes=head_b, flops=head_f)
    if kind == "step":  # + the logits once, and AdamW: p, m, v, g in and p, m, v out
        return dict(bytes=L * lay_b + 2 * 2.0 * V * H + 4.0 * T * V + 7 * 4.0 * L * LORA_LAYER,
                    flops=L * lay_f + head_f)
    nq, nkv = case["nq"], case["nkv"]
    n_in, n_out = T * HD * (nq + 2.0 * nkv), T * HD * (nq + 2.0 * nkv)
    if kind == "block":
        return dict(bytes=2 * n_in + 2.0 * T * nq * HD + 4 * n_out, flops=_causal(B, S, nq, 7))
    # the operators: q, k, v, o read by the backward again, dout fp32
    return dict(bytes=2 * 2 * n_in + 2 * 2.0 * T * nq * HD + 4.0 * T * nq * HD + 4 * n_out,
                flops=_causal(B, S, nq, 7))


def tolerance(case):
    # about four times the errors measured against 64 bits: a layer's adapter
    # gradients 7.8e-4 (fp16 operands and stashes, fp32 sums), the attention's dq
    # 4.1e-4, the whole step's adapter gradients 4.3e-3.  The head's dX 1e-5: its
    # fp16 operand rounds the small softmax entries, while the target's -1 is exact.
    return {"layer": {"rel": 3e-3}, "head": {"rel": 4e-5}, "block": {"rel": 1.7e-3},
            "attn": {"rel": 1.7e-3}, "step": {"rel": 1.8e-2}}[case["kind"]]


# ---------------------------------------------------------------- 64-bit reference

def _rms(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * w


def _rope(x):
    """Half-split rotation of x [B, S, n, 128]."""
    S = x.shape[1]
    d = torch.arange(HD // 2, device=x.device, dtype=torch.float64)
    ang = torch.arange(S, device=x.device, dtype=torch.float64)[:, None] * THETA ** (-2.0 * d / HD)
    c, s = ang.cos()[None, :, None], ang.sin()[None, :, None]
    a, b = x[..., :HD // 2], x[..., HD // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _attention(q, k, v):
    """(o [B, S, nq, 128], lse [B, nq, S]) of causal GQA attention, head by head group."""
    B, S, nq, _ = q.shape
    nkv = k.shape[2]
    mask = torch.ones(S, S, dtype=torch.bool, device=q.device).triu_(1)
    os_, ls = [], []
    for h in range(nq):
        kk, vv = k[:, :, h * nkv // nq], v[:, :, h * nkv // nq]
        s = q[:, :, h] @ kk.transpose(1, 2).contiguous() / math.sqrt(HD)
        s = s.masked_fill(mask, float("-inf"))
        l = torch.logsumexp(s, -1)
        os_.append(torch.exp(s - l[..., None]) @ vv)
        ls.append(l)
    return torch.stack(os_, 2), torch.stack(ls, 1)


def _split(flat, layers):
    out, at = [], 0
    for _ in range(layers):
        d = {}
        for n, o, i in PROJ:
            A = flat[at:at + R * i].view(R, i)
            at += R * i
            B = flat[at:at + o * R].view(o, R)
            at += o * R
            d[n] = (A, B)
        out.append(d)
    return out


def _layer64(x, ws, norms, ad, B, S):
    w = {}
    for (n, _, _), m in zip(MATS, ws):
        w[n] = m[0].double() * m[1].double()[:, None] if isinstance(m, tuple) else m.double()
    an, fn, qn, kn = (t.double() for t in norms)

    def lin(t, n):
        A, Bm = ad[n]
        return t @ w[n].t() + SCALE * ((t @ A.t()) @ Bm.t())

    xn = _rms(x, an)
    q = _rope(_rms(lin(xn, "wq").view(B, S, NQ, HD), qn))
    k = _rope(_rms(lin(xn, "wk").view(B, S, NKV, HD), kn))
    o, _ = _attention(q, k, lin(xn, "wv").view(B, S, NKV, HD))
    x = x + lin(o.reshape(B * S, Q), "wo")
    xn = _rms(x, fn)
    return x + (torch.nn.functional.silu(xn @ w["w_gate"].t()) * (xn @ w["w_up"].t())) @ w["w_down"].t()


def _ce64(logits, tgt):
    """Mean loss over the rows with a target inside their window."""
    B, S = tgt.shape
    lp = torch.log_softmax(logits.view(B, S, -1)[:, :-1], -1)
    return -lp.gather(2, tgt[:, :-1, None].long()).mean()


def exact(case, seed):
    g = _gen(seed)
    kind, B, S = case["kind"], case["B"], case["S"]
    if kind == "layer":
        ws, norms = _layer_weights(g, case["wfmt"])
        flat = _adapters(g, 1).double().requires_grad_()
        s = _inputs(case, g)
        x = s["x"].double().requires_grad_()
        y = _layer64(x, ws, norms, _split(flat, 1)[0], B, S)
        dx, dg = torch.autograd.grad(y, (x, flat), s["dy"].double())
        return dict(y=y.detach(), dx=dx, grads=dg)
    if kind == "head":
        E = _randn(g, (V, H), 0.02, torch.float16).double()
        s = _inputs(case, g)
        x = s["x"].double().requires_grad_()
        logits = x @ E.t()
        loss = _ce64(logits, s["tgt"])
        dl, dx = torch.autograd.grad(loss, (logits, x))
        return dict(loss=float(loss), dx=dx, dlogits=dl if case["dlogits"] else None)
    if kind == "step":
        frozen = [_layer_weights(g, case["wfmt"]) for _ in range(L)]
        E = _randn(g, (V, H), 0.02, torch.float16).double()
        fnorm = 1.0 + _randn(g, (H,), 0.1)
        flat = _adapters(g, L).double().requires_grad_()
        s = _inputs(case, g)
        x = E[s["tok"].reshape(-1).long()]
        ads = _split(flat, L)
        for l in range(L):
            x = torch.utils.checkpoint.checkpoint(_layer64, x, *frozen[l], ads[l], B, S,
                                                  use_reentrant=False)
        logits = _rms(x, fnorm.double()) @ E.t()
        loss = _ce64(logits, s["tgt"])
        dg, = torch.autograd.grad(loss, (flat,))
        return dict(loss=float(loss), logits=logits.detach(), grads=dg)
    s = _inputs(case, g)
    q, k, v = (s[n].double().requires_grad_() for n in "qkv")
    if kind == "block":
        o, _ = _attention(_rope(_rms(q, s["qn"].double())), _rope(_rms(k, s["kn"].double())), v)
        return torch.autograd.grad(o, (q, k, v), s["do"].double())
    o, lse = _attention(q, k, v)
    return (o.detach(), lse.detach()) + torch.autograd.grad(o, (q, k, v), s["do"].double())
