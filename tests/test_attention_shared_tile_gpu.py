"""Attention over 257 to 288 tokens: the ninth tile of 32, which a workgroup's eight wavefronts share (the queries of
the forward and of dQ, the keys of dK / dV) where there is no mask and the other axis has more than 192 tokens, and
the calls beside that rule, which the eight or four wavefronts take tile by tile (a causal mask, a short other axis, 256 tokens and
less), against the kernel oracle and torch's attention."""
import pytest
import torch

import test_kernels_gpu as base
from test_gemm_w4_gpu import hip, oracle  # noqa: F401  (fixtures)
from test_kernels_gpu import BF16, F16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("Tq,Tk,hd,causal", [
    (257, 257, 64, 0), (288, 288, 96, 0), (257, 288, 88, 1), (288, 257, 32, 0), (258, 1, 88, 0), (1, 258, 96, 0),
    (270, 40, 64, 0), (33, 270, 40, 1), (271, 271, 80, 1), (129, 160, 96, 0), (256, 256, 72, 1)])
def test_ninth_tile(hip, oracle, dtype, Tq, Tk, hd, causal):  # noqa: F811
    base.test_fused_attention(hip, oracle, dtype, dict(B=2, H=3, Tq=Tq, Tk=Tk, hd=hd, causal=causal, packed=False))


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("B,H,Tq,Tk,hd", [
    (2, 3, 257, 200, 64), (2, 3, 200, 257, 64), (2, 3, 288, 193, 96), (2, 3, 193, 288, 96), (2, 3, 257, 224, 88), (1, 3, 224, 288, 40),
    (3, 43, 257, 257, 88), (3, 43, 288, 288, 96), (3, 43, 257, 193, 80), (1, 129, 200, 260, 72)])
def test_shared_tile_sweeps(hip, oracle, dtype, B, H, Tq, Tk, hd):  # noqa: F811
    """Sweeps of 193 to 224 tokens leave the eighth wavefront without a tile (no maximum, no sum) and their operands take less
    LDS than the partial results; above head dim 64 dK / dV run on eight wavefronts, which share, for more than 128 heads only."""
    base.test_fused_attention(hip, oracle, dtype, dict(B=B, H=H, Tq=Tq, Tk=Tk, hd=hd, causal=0, packed=False))


@pytest.mark.parametrize("T,hd,causal", [(70, 64, 0), (130, 96, 1), (65, 128, 0)])
def test_tokens_far_apart(hip, T, hd, causal):  # noqa: F811
    """Token strides at which a tile's rows span more than 2 GiB (operands cut from one allocation of up to 8 GB) give what the
    same rows side by side give: every kernel sums alike in both forms, but for heads of up to 288 tokens side by side,
    which run in steps of 32 keys instead of 64 (fp32 sums of up to 130 products in another order, before results of
    16 bits: half a step of the type at most apart, twice where a second rounded value enters)."""
    H, st = 2, (1 << 30) // 128 + 8
    far = torch.zeros(4, T * st, dtype=BF16, device="cuda")
    near = [base.rnd((1, T, H, hd), BF16, i, 0.7).cuda() for i in range(4)]
    q, k, v, do = (torch.as_strided(far[i], (1, T, H, hd), (T * st, st, hd, 1)) for i in range(4))
    res = []
    for a, b, c, d in ((q, k, v, do), near):
        for dst, src in zip((a, b, c, d), near):
            dst.copy_(src)
        a, b, c, d = (x.permute(0, 2, 1, 3) for x in (a, b, c, d))
        o, dq, dk, dv = (torch.zeros(1, T, H, hd, dtype=BF16, device="cuda").permute(0, 2, 1, 3) for _ in range(4))
        lse, delta = torch.zeros(1, H, T, device="cuda"), torch.zeros(1, H, T, device="cuda")
        hip.run("attention_fwd", a, b, c, o, lse, hd ** -0.5, causal)
        hip.run("attention_bwd", a, b, c, o, d, lse, delta, dq, dk, dv, hd ** -0.5, causal)
        torch.cuda.synchronize()
        res.append([x.float().cpu() for x in (o, dq, dk, dv)])
    for x, y in zip(*res):
        torch.testing.assert_close(x, y, rtol=2.0 ** -7, atol=2.0 ** -8)
