"""GPU: row epilogues called on their own, against float64."""
import pytest
import torch

import llmt
import native

pytestmark = pytest.mark.gpu


def _norm_bwd_lora(L, dev, T, H, hscale, transposed=True):
    """The attention norm's backward on the LoRA input-gradient term alone (a
    zero GEMM row), (got, want): dh values of size hscale, in the GEMM's units."""
    g = torch.Generator().manual_seed(T + H)
    h = torch.randn(T, 48, generator=g) * hscale
    A = (torch.randn(48, H, generator=g) / H ** 0.5).half()
    x, w = torch.randn(T, H, generator=g), 1 + 0.1 * torch.randn(H, generator=g)
    rinv = torch.exp2(torch.randint(-20, 0, (T,), generator=g).float()) / hscale
    part = torch.cat([torch.zeros(T, H), h], 1).to(dev)
    Ad, At, xd, wd, rd = A.to(dev), A.t().contiguous().to(dev), x.to(dev), w.to(dev), rinv.to(dev)
    dh, out, ro = (torch.zeros(s, device=dev) for s in ((T, 64), (T, H), (T,)))
    g16 = torch.zeros(T, H, device=dev, dtype=torch.float16)
    p = lambda t: t.data_ptr()
    a = native.NormBwdArgs()
    r = a.inp
    r.part, r.split, r.ldp, r.hcol, r.nh, r.nterm, r.lscale = p(part), 1, H + 48, H, 48, 3, 2.0
    for q in range(3):
        t = r.term[q]
        t.shr, t.row0, t.kp, t.c0, t.n, t.hidx = p(Ad), 16 * q, H, 0, H, 16 * q
    a.rinv_in, a.gscale, a.dh_out, a.x, a.w, a.eps, a.H = p(rd), 1.0, p(dh), p(xd), p(wd), 1e-6, H
    a.dres_out, a.g16, a.rinv_out = p(out), p(g16), p(ro)
    a.lora_at = p(At) if transposed else None
    assert native.norm_bwd(L, a, T) == 0, L.llmt_last_error()
    torch.cuda.synchronize()
    d = 2.0 * (h.double() @ A.double()) * rinv.double()[:, None]
    xx, ww = x.double(), w.double()
    rr = torch.rsqrt((xx * xx).mean(1, keepdim=True) + 1e-6)
    want = rr * (d * ww - rr * rr / H * (d * ww * xx).sum(1, keepdim=True) * xx)
    return out.cpu(), want


@pytest.mark.parametrize("hscale", [1e-4, 3e3, 1e9])
@pytest.mark.parametrize("T,H,rows", [(200, 512, ""), (272, 512, ""), (520, 2048, ""),
                                      (784, 512, ""), (2064, 2048, ""), (49, 528, "8"),
                                      (784, 512, "no copy")])
def test_norm_bwd_lora_term_is_fp32(dev, L, monkeypatch, T, H, rows, hscale):
    """The LoRA input-gradient term at every rows-a-workgroup count (1, 2, 3
    and 4 by the token count, 8 by the override; one without the transposed
    adapter copy), for dh values of any size.  Bound: the 48 products and their sum, the row factor
    and the few operations after it, each 2^-24: 60 * 2^-24 = 3.6e-6, row by
    row (the rows' factors differ by 2^20)."""
    print(f"case: norm_bwd LoRA term T{T} H{H} rows {rows or 'by T'} dh {hscale:g}", flush=True)
    monkeypatch.setenv("LLMT_ROWS_PER_WG", rows if rows.isdigit() else "")
    got, want = _norm_bwd_lora(L, dev, T, H, hscale, rows != "no copy")
    err = ((got.double() - want).norm(dim=1) / want.norm(dim=1)).max()
    assert float(err) < 3.6e-6
