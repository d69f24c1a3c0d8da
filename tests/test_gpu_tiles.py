"""GPU: the GEMM tiles at the row counts where they change (edges of the 32-,
64-, 128- and 256-row tiles, remainders of all of them), with fp16 and int8
weights: the standalone products, one full-width decoder layer (the Q/K/V and
O GEMMs' LoRA rows, the SwiGLU epilogue, the per-k scales of int8 dX GEMMs)
against the fp32 oracle, and the head with its softmax statistics."""
import numpy as np
import pytest
import torch

import llmt
import native
from helpers import grad_errors, rel_l2
from oracle import lora_step as ref
from oracle.configs import make_adapters, make_layer
from oracle.quant import quantize_rows

pytestmark = pytest.mark.gpu

GRAD_TOL = 1e-2


@pytest.mark.parametrize("i8", [False, True])
@pytest.mark.parametrize("M", [16, 48, 80, 144, 336, 528, 1040])
@pytest.mark.parametrize("N,K", [(16, 64), (176, 192), (2064, 2048), (4096, 320)])
def test_gemm_row_tiles(dev, L, i8, M, N, K):
    # fp16 operands (int8 ones are exact in fp16), fp32 sums of K products in
    # another order: 1e-5 is the bar of the other GEMM tests
    print(f"case: gemm i8={i8} M{M} N{N} K{K}", flush=True)
    g = torch.Generator().manual_seed(M + N + K)
    A = torch.randn(M, K, generator=g).half()
    w = torch.randn(N, K, generator=g) * 0.02
    if i8:
        q, sc = quantize_rows(w.numpy())
        sc16 = torch.from_numpy(sc.astype(np.float16))
        qt = torch.from_numpy(q)
        want = (A.float() @ qt.float().t()) * sc16.float()[None, :]
        got = llmt.gemm_i8(A.to(dev), qt.to(dev), sc16.to(dev)).cpu()
    else:
        B = w.half()
        want = A.float() @ B.float().t()
        got = llmt.gemm_f16(A.to(dev), B.to(dev)).cpu()
    assert rel_l2(got, want) < 1e-5
    assert torch.isfinite(got).all()


def _off(t, n=1):
    """t's values in memory that starts n elements past a 16-byte boundary."""
    return torch.cat([t.new_zeros(n), t.reshape(-1)])[n:].view(t.shape)


@pytest.mark.parametrize("i8", [False, True])
@pytest.mark.parametrize("M", [16, 48, 96, 128, 1040])
def test_gemm_unaligned_rows(dev, L, i8, M):
    """A that does not start on a 16-byte boundary (2, 4 and 8 bytes past it):
    the register-staged kernel, every row form of it, fp32 sums in its own
    order against the aligned call."""
    print(f"case: gemm unaligned i8={i8} M{M}", flush=True)
    N, K = 176, 320
    g = torch.Generator().manual_seed(M)
    A = torch.randn(M, K, generator=g).half().to(dev)
    if i8:
        q, sc = quantize_rows((torch.randn(N, K, generator=g) * 0.02).numpy())
        q, sc = torch.from_numpy(q).to(dev), torch.from_numpy(sc.astype(np.float16)).to(dev)
        run = lambda a: llmt.gemm_i8(a, q, sc)
    else:
        B = (torch.randn(N, K, generator=g) * 0.02).half().to(dev)
        run = lambda a: llmt.gemm_f16(a, B)
    want = run(A).cpu()
    for n in (1, 2, 4):
        a = _off(A, n)
        assert a.data_ptr() % 16 == 2 * n
        assert rel_l2(run(a).cpu(), want) < 1e-5


@pytest.mark.parametrize("T", [16, 48, 128, 1040])
def test_head_unaligned_rows(dev, T):
    """The head on hidden states off a 16-byte boundary against the aligned
    call: the same logits up to the order of their sums."""
    print(f"case: head unaligned T{T}", flush=True)
    H, V = 512, 2496
    g = torch.Generator().manual_seed(T)
    E = (torch.randn(V, H, generator=g) * 0.05).half().to(dev)
    x = torch.randn(T, H, generator=g).half().to(dev)
    tgt = torch.randint(0, V, (1, T), generator=g, dtype=torch.int32).to(dev)
    d = ref.Dims(**{**ref.QWEN3_1_7B.__dict__, "n_layers": 1, "vocab": V, "hidden": H,
                    "intermediate": 512, "n_heads": 2, "n_kv_heads": 1})
    ctx = llmt.Context(llmt.make_dims(d), 1, T)
    try:
        ctx.set_embed_f16(E, torch.ones(H, device=dev))
        loss, dl, dx = (t.cpu() if torch.is_tensor(t) else t
                        for t in ctx.head_ce(x, tgt, want_dlogits=True))
        loss2, dl2, dx2 = ctx.head_ce(_off(x), tgt, want_dlogits=True)
        assert abs(loss2 - loss) < 1e-4
        assert rel_l2(dl2.cpu(), dl) < 1e-4 and rel_l2(dx2.cpu(), dx) < 1e-3
    finally:
        ctx.close()


DMA_KINDS = {(False, 1040): {"gu"}, (True, 1040): {"gu"}, (True, 1424): {"gudx"},
             (False, 2000): {"qkv"}, (True, 2000): {"qkv"},
             (False, 4080): {"qkv", "o", "gu", "gudx", "odx", "qkvdx"},
             (True, 4080): {"qkv", "o", "gu", "odx", "qkvdx"}}


@pytest.mark.parametrize("int8,B,S", [(False, 1, 16), (False, 1, 80), (False, 3, 208),
                                      (False, 5, 400), (True, 1, 48), (True, 1, 208),
                                      (True, 1, 336), (True, 5, 400), (True, 1, 16),
                                      (True, 1, 80), (False, 2, 520), (True, 2, 520),
                                      (True, 2, 712), (False, 8, 510), (True, 8, 510)])
def test_layer_row_tiles_match_oracle(dev, L, int8, B, S):
    """From 1040 rows the plan takes 256-row tiles for some of the GEMMs, with
    ragged last row blocks here; DMA_KINDS says which, so that a case does not
    quietly come to test another kernel."""
    print(f"case: full-width layer int8={int8} B{B} S{S}", flush=True)
    d = ref.Dims(**{**ref.QWEN3_1_7B.__dict__, "n_layers": 1, "vocab": 256})
    plan = native.layer_plan(L, d, B * S, int8)
    assert {n for n, k in plan.items() if k.startswith("gemm_dma")} == DMA_KINDS.get(
        (int8, B * S), set()), plan
    g = torch.Generator().manual_seed(B * 1000 + S)
    lw = make_layer(g, d)
    ad = make_adapters(g, d)[0]
    x, dy = torch.randn(B * S, d.hidden, generator=g), torch.randn(B * S, d.hidden, generator=g)
    names = ("wq", "wk", "wv", "wo", "w_gate", "w_up", "w_down")
    f = lambda t: t.to(torch.float32).to(dev).contiguous()
    norms = [f(t) for t in (lw.attn_norm, lw.ffn_norm, lw.q_norm, lw.k_norm)]
    ctx = llmt.Context(llmt.make_dims(d), B, S, int8=int8)
    try:
        if int8:
            qs, ss = [], []
            for n in names:
                q, sc = quantize_rows(getattr(lw, n).float().numpy())
                sc16 = sc.astype(np.float16)
                qs.append(torch.from_numpy(q).to(dev))
                ss.append(torch.from_numpy(sc16).to(dev))
                setattr(lw, n, torch.from_numpy(q.astype(np.float32) *
                                                sc16.astype(np.float32)[:, None]))
            ctx.set_layer_i8(0, qs, ss, *norms)
        else:
            ctx.set_layer_f16(0, *(getattr(lw, n).half().to(dev).contiguous() for n in names), *norms)
        cos, sin = ref.rope_tables(S, d.head_dim, d.theta)
        y_ref, st = ref.layer_forward(x, lw, ad, d, B, S, cos, sin)
        dx_ref, grads_ref = ref.layer_backward(dy, st, lw, ad, d, B, S, cos, sin)
        ctx.lora_set("param", llmt.flatten_adapters([ad]).to(dev))
        y = ctx.layer_forward(0, x.to(dev), B)
        assert rel_l2(y.cpu(), y_ref) < GRAD_TOL
        dx = ctx.layer_backward(0, dy.to(dev), B)
        assert rel_l2(dx.cpu(), dx_ref) < GRAD_TOL
        errs = grad_errors(ctx.lora_get("grad"), [grads_ref], d)
        print("worst", max(errs.items(), key=lambda kv: kv[1]), flush=True)
        assert max(errs.values()) < GRAD_TOL
    finally:
        ctx.close()


@pytest.mark.parametrize("T", [16, 48, 112, 336, 528, 1040])
def test_head_row_tiles(dev, T):
    print(f"case: head T{T}", flush=True)
    H, V = 512, 9984  # 78 tiles of 128 columns, 39 of 256, 52 of 192
    g = torch.Generator().manual_seed(T)
    E = (torch.randn(V, H, generator=g) * 0.05).half()
    x = torch.randn(T, H, generator=g).half()
    tgt = torch.randint(0, V, (T,), generator=g, dtype=torch.int32)
    logits = x.float() @ E.float().t()
    loss_ref, dl_ref, _ = ref.cross_entropy(logits, tgt, ref.valid_rows(1, T))
    d = ref.Dims(**{**ref.QWEN3_1_7B.__dict__, "n_layers": 1, "vocab": V, "hidden": H,
                    "intermediate": 512, "n_heads": 2, "n_kv_heads": 1})
    ctx = llmt.Context(llmt.make_dims(d), 1, T)
    try:
        ctx.set_embed_f16(E.to(dev), torch.ones(H, device=dev))
        loss, dl, dx = ctx.head_ce(x.to(dev), tgt.view(1, T).to(dev), want_dlogits=True)
        assert abs(loss - float(loss_ref)) < 1e-3
        assert rel_l2(dl.cpu(), dl_ref) < 1e-4
        assert rel_l2(dx.cpu(), dl_ref @ E.float()) < 1e-3
    finally:
        ctx.close()


def _small_layer_matches_oracle(dev, d, B, S, **adapter_kw):
    """Forward, dx and adapter gradients of one fp16 layer."""
    T = B * S
    g = torch.Generator().manual_seed(T)
    lw = make_layer(g, d)
    ad = make_adapters(g, d, **adapter_kw)[0]
    x, dy = torch.randn(T, d.hidden, generator=g), torch.randn(T, d.hidden, generator=g)
    f = lambda t: t.to(torch.float32).to(dev).contiguous()
    cos, sin = ref.rope_tables(S, d.head_dim, d.theta)
    y_ref, st = ref.layer_forward(x, lw, ad, d, B, S, cos, sin)
    dx_ref, grads_ref = ref.layer_backward(dy, st, lw, ad, d, B, S, cos, sin)
    ctx = llmt.Context(llmt.make_dims(d), B, S)
    try:
        ctx.set_layer_f16(0, *(getattr(lw, n).half().to(dev).contiguous() for n in
                               ("wq", "wk", "wv", "wo", "w_gate", "w_up", "w_down")),
                          f(lw.attn_norm), f(lw.ffn_norm), f(lw.q_norm), f(lw.k_norm))
        ctx.lora_set("param", llmt.flatten_adapters([ad]).to(dev))
        assert rel_l2(ctx.layer_forward(0, x.to(dev), B).cpu(), y_ref) < GRAD_TOL
        assert rel_l2(ctx.layer_backward(0, dy.to(dev), B).cpu(), dx_ref) < GRAD_TOL
        errs = grad_errors(ctx.lora_get("grad"), [grads_ref], d)
        assert max(errs.values()) < GRAD_TOL
    finally:
        ctx.close()


@pytest.mark.parametrize("T", [16, 272, 528, 784])
def test_layer_row_epilogues_at_row_counts(dev, T):
    """One small layer at token counts on both sides of the row epilogues'
    rows-a-workgroup steps (256, 512, 768 rows), adapters large enough for
    their input-gradient term (three fp16 parts of dh on the matrix cores
    above 256 rows) to dominate dx."""
    print(f"case: row epilogues T{T}", flush=True)
    d = ref.Dims(**{**ref.QWEN3_1_7B.__dict__, "n_layers": 1, "vocab": 256, "hidden": 512,
                    "intermediate": 512, "n_heads": 4, "n_kv_heads": 2})
    _small_layer_matches_oracle(dev, d, 1, T, b_std=0.5)


@pytest.mark.parametrize("S", [500, 512])
def test_layer_last_wave_split(dev, L, S):
    """A layer whose down-projection dX (N = intermediate, K = hidden) ends in a
    partial wave of 256 x 256 tiles, which the plan then splits over K: whole
    and ragged row blocks, read by the SwiGLU backward."""
    print(f"case: last-wave split B16 S{S}", flush=True)
    d = ref.Dims(**{**ref.QWEN3_1_7B.__dict__, "n_layers": 1, "vocab": 256, "hidden": 512,
                    "intermediate": 4352, "n_heads": 2, "n_kv_heads": 1})
    assert 0 < native.gemm_split_col(L, 16 * S, d.intermediate, d.hidden, False) < d.intermediate
    _small_layer_matches_oracle(dev, d, 16, S)


@pytest.mark.parametrize("T,H", [(16, 512), (48, 2048), (32, 2112)])
def test_layer_input_alignment(dev, T, H):
    """The layer API's row passes on inputs that start off a 16-byte boundary
    (and on rows wider than 2048 columns) against the aligned call: the same
    values, so the fp32 outputs agree to the rounding of an fp16 operand."""
    print(f"case: layer input alignment T{T} H{H}", flush=True)
    d = ref.Dims(**{**ref.QWEN3_1_7B.__dict__, "n_layers": 1, "vocab": 256, "hidden": H,
                    "intermediate": 256, "n_heads": 2, "n_kv_heads": 1})
    g = torch.Generator().manual_seed(T + H)
    lw = make_layer(g, d)
    ad = make_adapters(g, d)[0]
    f = lambda t: t.to(torch.float32).to(dev).contiguous()
    ctx = llmt.Context(llmt.make_dims(d), 1, T)
    try:
        ctx.set_layer_f16(0, *(getattr(lw, n).half().to(dev).contiguous() for n in
                               ("wq", "wk", "wv", "wo", "w_gate", "w_up", "w_down")),
                          f(lw.attn_norm), f(lw.ffn_norm), f(lw.q_norm), f(lw.k_norm))
        ctx.lora_set("param", llmt.flatten_adapters([ad]).to(dev))
        x, dy = torch.randn(T, H, generator=g).to(dev), torch.randn(T, H, generator=g).to(dev)
        y, dx = ctx.layer_forward(0, x, 1), ctx.layer_backward(0, dy, 1)
        y2, dx2 = ctx.layer_forward(0, _off(x), 1), ctx.layer_backward(0, _off(dy), 1)
        assert rel_l2(y2.cpu(), y.cpu()) < 1e-3 and rel_l2(dx2.cpu(), dx.cpu()) < 1e-3
    finally:
        ctx.close()


@pytest.mark.parametrize("B,S,nq,nkv", [(1, 33, 16, 8), (2, 47, 8, 8), (1, 250, 32, 8),
                                        (1, 530, 16, 8), (3, 333, 16, 8), (2, 700, 16, 8),
                                        (1, 1100, 8, 4)])
def test_attention_grid_sizes(dev, B, S, nq, nkv):
    """The attention backward on both sides of its small-grid rule (16-key
    blocks split over four waves in 32-query tiles, then one launch, then
    two), ragged S, through the operators and the fused block."""
    print(f"case: attention B{B} S{S} nq{nq} nkv{nkv}", flush=True)
    g = torch.Generator().manual_seed(3 * S + nq)
    q = torch.randn(B, S, nq, 128, generator=g).half()
    k = torch.randn(B, S, nkv, 128, generator=g).half()
    v = torch.randn(B, S, nkv, 128, generator=g).half()
    do = torch.randn(B, S, nq, 128, generator=g)
    o_ref, lse_ref = ref.attention_fwd(q.float(), k.float(), v.float())
    qd, kd, vd = q.to(dev), k.to(dev), v.to(dev)
    o, lse = llmt.attention_fwd(qd, kd, vd)
    assert rel_l2(o.float().cpu(), o_ref) < 2e-3
    assert (lse.cpu() - lse_ref).abs().max() < 1e-3
    want = ref.attention_bwd(do, q.float(), k.float(), v.float(), o.float().cpu(), lse.cpu())
    for a, b in zip(llmt.attention_bwd(qd, kd, vd, o, lse, do.to(dev)), want):
        assert rel_l2(a.cpu(), b) < GRAD_TOL
    # the block on inputs whose norm and rotation the oracle applies
    cos, sin = ref.rope_tables(S, 128, 1e6)
    one = torch.ones(128)
    rot = lambda t: ref.rope_fwd(ref.rmsnorm(t.float(), one, 1e-6), cos, sin)
    x = [t.float().requires_grad_() for t in (q, k)]
    with torch.enable_grad():
        qr, kr = (rot(t) for t in x)
    od, ld = ref.attention_fwd(qr.detach(), kr.detach(), v.float())
    dqr, dkr, dv_ref = ref.attention_bwd(do.half().float(), qr.detach(), kr.detach(), v.float(), od, ld)
    dq_ref, dk_ref = torch.autograd.grad((qr, kr), x, (dqr, dkr))
    got = llmt.attention_block_bwd(qd, kd, vd, one.to(dev), one.to(dev), do.half().to(dev))
    for a, b in zip(got, (dq_ref, dk_ref, dv_ref)):
        assert rel_l2(a.cpu(), b) < GRAD_TOL


@pytest.mark.parametrize("B,S,nq,nkv", [(1, 1, 16, 8), (1, 17, 4, 1), (2, 31, 16, 8), (1, 129, 16, 8),
                                        (1, 512, 16, 8), (1, 513, 16, 8), (2, 272, 16, 8),
                                        (3, 257, 8, 8), (2, 530, 16, 8), (1, 1061, 16, 8),
                                        (1, 2061, 4, 2), (1, 2061, 24, 3)])
def test_attention_forward_key_split(dev, B, S, nq, nkv):
    """The attention forward on both sides of its rule: keys split over the
    waves of 16- and of 32-query workgroups, then one sweep a wave; ragged S,
    fewer key tiles than waves.  A NaN query row stays in its own row."""
    print(f"case: attention forward B{B} S{S} nq{nq} nkv{nkv}", flush=True)
    g = torch.Generator().manual_seed(5 * S + nq)
    q = torch.randn(B, S, nq, 128, generator=g).half()
    k = torch.randn(B, S, nkv, 128, generator=g).half()
    v = torch.randn(B, S, nkv, 128, generator=g).half()
    o_ref, lse_ref = ref.attention_fwd(q.float(), k.float(), v.float())
    o, lse = llmt.attention_fwd(q.to(dev), k.to(dev), v.to(dev))
    # fp16 probabilities and output: 2^-11 each, at most a few of them a row
    assert rel_l2(o.float().cpu(), o_ref) < 2e-3
    assert (lse.cpu() - lse_ref).abs().max() < 1e-3
    r = S // 2
    q[:, r, 0] = float("nan")
    o2, lse2 = llmt.attention_fwd(q.to(dev), k.to(dev), v.to(dev))
    assert torch.isnan(o2[:, r, 0]).all() and torch.isnan(lse2[:, 0, r]).all()
    o2[:, r, 0], lse2[:, 0, r] = o[:, r, 0], lse[:, 0, r]
    assert torch.equal(o2, o) and torch.equal(lse2, lse)


@pytest.mark.parametrize("B,S,nq,nkv", [(1, 431, 16, 8), (1, 450, 16, 8), (2, 799, 8, 4),
                                        (1, 1063, 8, 1), (4, 1030, 4, 4), (1, 770, 1, 1),
                                        (1, 2033, 2, 1), (1, 767, 4, 4), (4, 1217, 4, 4)])
def test_attention_backward_key_split(dev, B, S, nq, nkv):
    """The dQ blocks whose keys are split over the waves (few heads), ragged
    last blocks: 328 to 1312 workgroups by the rule's count; below 320 from S =
    768 with at most two query heads a KV head (62 and 192).  Beside them what
    the rule leaves to the other forms: 203 workgroups at 8 / 1, S = 767, and
    1552 workgroups."""
    test_attention_grid_sizes(dev, B, S, nq, nkv)
