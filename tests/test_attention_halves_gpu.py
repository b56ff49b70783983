"""Backward of short heads: heads in one workgroup and heads in two give the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Tq,Tk,hd,causal", [(197, 197, 64, 0), (129, 129, 64, 1), (256, 256, 64, 1), (40, 250, 32, 0), (225, 7, 48, 0), (161, 255, 56, 1)])
def test_heads_in_halves(Tq, Tk, hd, causal):
    """400 heads: 256 and 144, all whole; 260: 256 whole and four in halves; the four alone.  Gradients of the last four in all three."""
    from pfeife_amd.hip import HipKernels

    hip = HipKernels()
    g = torch.Generator().manual_seed(Tq + Tk)
    n = 400
    mk = lambda T: torch.randn(n, 1, T, hd, generator=g).to(torch.bfloat16).cuda()
    q, k, v, d_o = mk(Tq), mk(Tk), mk(Tk), mk(Tq)
    o, lse = torch.zeros_like(q), torch.zeros(n, 1, Tq, device="cuda")
    hip.run("attention_fwd", q, k, v, o, lse, hd ** -0.5, causal)
    got = []
    for heads in (slice(0, 400), slice(140, 400), slice(396, 400)):
        outs = [torch.full_like(t[heads], 7.0) for t in (q, k, v)]
        delta = torch.full_like(lse[heads], 7.0)
        hip.run("attention_bwd", q[heads], k[heads], v[heads], o[heads], d_o[heads], lse[heads], delta, *outs, hd ** -0.5, causal)
        torch.cuda.synchronize()
        got.append([t[-4:] for t in outs] + [delta[-4:]])
    for other in got[1:]:
        for a, b in zip(got[0], other):
            assert torch.equal(a, b)
    # what both give, against 64 bits (the bound of the 16-bit attention tests)
    qd, kd, vd, dd = (t[396:].double() for t in (q, k, v, d_o))
    s = qd @ kd.transpose(2, 3).contiguous() * hd ** -0.5
    if causal:
        s = s.masked_fill(torch.ones(Tq, Tk, dtype=torch.bool, device="cuda").triu(1 + Tk - Tq), -torch.inf)
    p = s.softmax(-1)
    dp = dd @ vd.transpose(2, 3).contiguous()
    ds = p * (dp - (p * dp).sum(-1, keepdim=True)) * hd ** -0.5
    for a, want in zip(got[0], (ds @ kd, ds.transpose(2, 3).contiguous() @ qd, p.transpose(2, 3).contiguous() @ dd)):
        assert float((a.double() - want).norm() / want.norm()) <= 2e-2
