"""delta = rowsum(dO * O) of the tiled attention backward: as near to 64 bits as short chains of fp32 sums are."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def chains(x, y):
    """Sums of eight products each, one after the other as fused multiply-adds round them, then neighbours in pairs: [..., hd] -> [...] in fp32."""
    s = torch.zeros(x.shape[:-1] + (x.shape[-1] // 8,), dtype=torch.float32)
    x, y = (t.double().unflatten(-1, (-1, 8)) for t in (x, y))
    for k in range(8):
        s = (s.double() + x[..., k] * y[..., k]).float()
    part = list(s.unbind(-1))
    while len(part) > 1:
        part = [a + b for a, b in zip(part[::2], part[1::2])] + part[len(part) // 2 * 2:]
    return part[0]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hd,Tq,Tk,causal", [(32, 320, 320, 1), (64, 333, 333, 0), (64, 1024, 77, 0), (80, 320, 500, 0), (96, 513, 513, 1),
                                             (128, 320, 320, 1)])
def test_delta_is_as_exact_as_chains_of_eight(hip, hd, Tq, Tk, causal, dtype):
    B, H = 1, 3
    g = torch.Generator().manual_seed(hd + Tq)
    token_major = lambda t: torch.randn(B, t, H, hd, generator=g).to(dtype).cuda().permute(0, 2, 1, 3)
    q, k, v, do = token_major(Tq), token_major(Tk), token_major(Tk), token_major(Tq)
    o, dq, dk, dv = (torch.zeros_like(t) for t in (q, q, k, v))
    o_lo = torch.zeros_like(q) if hd > hip.O_LO_HEAD_DIM else None
    lse, delta = torch.zeros(B, H, Tq, device="cuda"), torch.zeros(B, H, Tq, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    hip.attention_fwd(q, k, v, o, lse, hd ** -0.5, causal, o_lo)(s)
    hip.attention_bwd(q, k, v, o, do, lse, delta, dq, dk, dv, hd ** -0.5, causal, o_lo)(s)
    torch.cuda.synchronize()
    O = o.float().cpu() if o_lo is None else o.float().cpu() + o_lo.float().cpu() / 2048
    exact = (O.double() * do.double().cpu()).sum(-1)
    pad = lambda t: torch.nn.functional.pad(t, (0, -hd % 16))
    error, short = ((t.double() - exact).norm() for t in (delta.cpu(), chains(pad(O), pad(do.float().cpu()))))
    assert short > 0 and error <= 1.1 * short      # (one chain of a half row, in fp16: 1.5 times as much at 64, 1.9 at 128)
