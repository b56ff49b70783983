"""Norms of rows that share a wavefront (up to 512 columns): widths and row counts at the edges, against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from pfeife_amd.hip import HipKernels
    return HipKernels()


def guarded(rows, d, dtype):
    """A result with a border that must stay as it is."""
    t = torch.full((rows * d + 16,), 7.0, dtype=dtype, device="cuda")
    return t, t[:rows * d].view(rows, d)


@pytest.mark.parametrize("io,lp", [(torch.float32, torch.bfloat16), (torch.float32, torch.float16), (torch.float16, None), (torch.bfloat16, None)])
@pytest.mark.parametrize("rows,d,rms", [(1, 8, False), (65, 64, True), (2300, 72, False), (31, 128, False), (4100, 136, True), (17, 256, False),
                                        (2049, 264, False), (1023, 384, True), (4099, 512, False)])
def test_narrow_norms(hip, io, lp, rows, d, rms):
    """Bound: `d` units of roundoff of what a row's sums hold in magnitudes, `rows` of what a column's do, and a rounding of the result."""
    g = torch.Generator().manual_seed(rows + d)
    rnd = lambda *s: torch.randn(*s, generator=g).cuda()
    dy_dt = lp or io
    x, dy, add = (rnd(rows, d) + 0.3).to(io), rnd(rows, d).to(dy_dt), rnd(rows, d).to(io)
    gamma, beta = rnd(d) + 1, rnd(d)
    u = lambda dt: {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dt]
    xd = x.double()
    mu = torch.zeros(rows, 1, device="cuda", dtype=torch.float64) if rms else xd.mean(1, keepdim=True)
    rs = 1 / ((xd - mu).square().mean(1, keepdim=True) + 1e-5).sqrt()
    xh = (xd - mu) * rs
    # forward
    whole, y = guarded(rows, d, dy_dt)
    mean, rstd = torch.zeros(rows, device="cuda"), torch.zeros(rows, device="cuda")
    if rms:
        hip.run("rmsnorm_fwd", x, gamma, y, rstd, rows, d, 1e-5)
    else:
        hip.run("layernorm_fwd", x, gamma, beta, y, mean, rstd, rows, d, 1e-5)
    torch.cuda.synchronize()
    eps = (d + 8) * 2.0 ** -24
    want = xh * gamma + (0 if rms else beta)
    size = (xd.abs() + xd.abs().mean(1, keepdim=True)) * rs * (1 + xh.abs())
    assert ((rstd.double() - rs[:, 0]).abs() <= eps * rs[:, 0] * (1 + (xd.square().mean(1) * rs[:, 0] ** 2))).all()
    assert ((y.double() - want).abs() <= eps * (size * gamma.abs() + want.abs() + 1) + u(dy_dt) * want.abs()).all()
    assert (whole[rows * d:] == 7).all()
    # backward, with the 16-bit copy and its column sums or with everything in 16 bits
    whole_dx, dx = guarded(rows, d, io)
    dyd = dy.double()
    gg = dyd * gamma
    c1 = torch.zeros_like(mu) if rms else gg.mean(1, keepdim=True)
    want = rs * (gg - c1 - xh * (gg * xh).mean(1, keepdim=True)) + add.double()
    m = rs * (gg.abs() + gg.abs().mean(1, keepdim=True) + (xh.abs() + size) * (gg * xh).abs().mean(1, keepdim=True)) + add.double().abs()
    nb = hip.norm_bwd_partials(rows)
    kinds = 3 if lp else 2
    ws = torch.full((nb * kinds * d + 16,), 7.0, device="cuda")
    mean_, rstd_ = (None if rms else mu[:, 0].float()), rs[:, 0].float()
    if lp:
        whole_lp, dx_lp = guarded(rows, d, lp)
        hip.run("norm_bwd_fused", dy, x, gamma, mean_, rstd_, add, dx, dx_lp, ws, rows, d, True, True)
    elif rms:
        hip.run("rmsnorm_bwd", dy, x, gamma, rstd_, add, dx, torch.zeros(d, device="cuda"), ws, rows, d, 1)
    else:
        hip.run("layernorm_bwd", dy, x, gamma, mean_, rstd_, add, dx, torch.zeros(d, device="cuda"), torch.zeros(d, device="cuda"), ws, rows, d, 1)
    torch.cuda.synchronize()
    assert ((dx.double() - want).abs() <= 4 * eps * m + u(io) * want.abs()).all()
    assert (whole_dx[rows * d:] == 7).all() and (ws[nb * kinds * d:] == 7).all()
    part = ws[:nb * kinds * d].view(nb, kinds, d).double().sum(0)
    room = (rows + 16) * 2.0 ** -24
    assert ((part[0] - (dyd * xh).sum(0)).abs() <= room * (dyd.abs() * (xh.abs() + size)).sum(0) + 1e-30).all()
    assert ((part[1] - dyd.sum(0)).abs() <= room * dyd.abs().sum(0) + 1e-30).all()
    if lp:
        assert torch.equal(dx_lp, dx.to(lp)) and (whole_lp[rows * d:] == 7).all()
        assert ((part[2] - dx_lp.double().sum(0)).abs() <= room * dx_lp.double().abs().sum(0) + 1e-30).all()
