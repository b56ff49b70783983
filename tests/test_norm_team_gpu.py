"""Norm backward of rows of 513 to 2048 columns (a team of wavefronts to a row) at its edges, against the kernel oracle:
columns that fill no wavefront, rows that fill no workgroup, one row and many."""
import pytest
import torch

from test_kernels_gpu import BF16, F16, F32, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dy_dt,io_dt,lp_dt", [(F16, F32, F16), (BF16, F32, BF16), (F32, F32, None), (F32, F32, BF16), (BF16, BF16, None)])
@pytest.mark.parametrize("rows,d", [(1, 520), (3, 1024), (5, 1032), (513, 1408), (8, 1536), (2051, 1544), (700, 2048), (4097, 768)])
def test_against_the_oracle(rows, d, dy_dt, io_dt, lp_dt):
    from oracle.kernels_oracle import OracleKernels
    from pfeife_amd.hip import HipKernels

    hip, oracle = HipKernels(0), OracleKernels("cpu")
    for rms, add_in_place in ((False, False), (True, True)):
        x, dy, add = rnd((rows, d), io_dt, 1), rnd((rows, d), dy_dt, 2), rnd((rows, d), io_dt, 3)
        gamma, mean, rstd = rnd((d,), F32, 4), rnd((rows,), F32, 5) * 0.1, rnd((rows,), F32, 6).abs() + 0.5
        out = {}
        for k, dev in ((hip, "cuda"), (oracle, "cpu")):
            t = {n: v.clone().to(dev) for n, v in dict(x=x, dy=dy, add=add, g=gamma, m=mean, r=rstd).items()}
            dx = t["add"] if add_in_place else torch.zeros(rows, d, dtype=io_dt, device=dev)
            m = None if rms else t["m"]
            lp = None if lp_dt is None else torch.zeros(rows, d, dtype=lp_dt, device=dev)
            if lp is not None:
                nb = k.norm_bwd_partials(rows)
                ws = torch.zeros(nb * 3 * d, device=dev)
                k.norm_bwd_fused(t["dy"], t["x"], t["g"], m, t["r"], t["add"], dx, lp, ws, rows, d, True, True)(
                    torch.cuda.current_stream().cuda_stream)
                sums = ws.view(nb, 3, d).double().sum(0)
            else:
                nb = k.norm_bwd_partials(rows)
                ws = torch.zeros(max(k.colreduce_workspace(rows, d), 2 * d * nb), device=dev)
                fn = (k.rmsnorm_bwd(t["dy"], t["x"], t["g"], t["r"], t["add"], dx, None, ws, rows, d, defer=1) if rms else
                      k.layernorm_bwd(t["dy"], t["x"], t["g"], m, t["r"], t["add"], dx, None, None, ws, rows, d, defer=1))
                fn(torch.cuda.current_stream().cuda_stream)
                sums = ws[:nb * 2 * d].view(nb, 2, d).double().sum(0)
            out[dev] = (dx.cpu(), None if lp is None else lp.cpu(), sums.cpu())
        torch.cuda.synchronize()
        (a, al, asum), (b, bl, bsum) = out["cuda"], out["cpu"]
        rt = {F32: 2e-5, F16: 4e-3, BF16: 2e-2}
        torch.testing.assert_close(a.float(), b.float(), rtol=rt[io_dt], atol=rt[io_dt] * 4)
        if al is not None:
            torch.testing.assert_close(al.float(), bl.float(), rtol=rt[lp_dt], atol=rt[lp_dt] * 4)
        # fp32 sums of `rows` terms each, in another order; a side copy rounded the other way shifts its column sum by one ulp of it
        scale = float(bsum.abs().max()) + 1.0
        tol = rows * 2.0 ** -24 * scale + (0 if al is None else float((al.float() - bl.float()).abs().sum(0).max()))
        assert float((asum[:2] - bsum[:2]).abs().max()) <= rows * 2.0 ** -24 * scale + 1e-4 * scale
        if al is not None:
            assert float((asum[2] - bsum[2]).abs().max()) <= tol + 1e-4 * scale


@pytest.mark.parametrize("rows,d", [(64, 1024), (33, 2048)])
def test_non_finite_rows_stay_in_their_rows(rows, d):
    """A row of infinities gives NaN in that row only."""
    from pfeife_amd.hip import HipKernels

    hip = HipKernels(0)
    dy, x = rnd((rows, d), BF16, 1).cuda(), rnd((rows, d), F32, 2).cuda()
    dy[7] = float("inf")
    dx, lp = torch.zeros(rows, d, device="cuda"), torch.zeros(rows, d, dtype=BF16, device="cuda")
    ws = torch.zeros(hip.norm_bwd_partials(rows) * 2 * d, device="cuda")
    hip.norm_bwd_fused(dy, x, torch.ones(d, device="cuda"), torch.zeros(rows, device="cuda"), torch.ones(rows, device="cuda"), None, dx, lp,
                       ws, rows, d, True, False)(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    bad = ~torch.isfinite(dx).all(dim=1)
    assert bad.nonzero().flatten().tolist() == [7]


@pytest.mark.parametrize("rows,d", [(5, 520), (700, 1408), (300, 2048)])
def test_partial_rows_at_any_fp32_address(rows, d):
    """The workspace needs no more than its type's alignment: the partial rows are the same sums at every offset (of at
    most `rows` fp32 terms, in another order: rows * 2^-24 of the sum of their magnitudes)."""
    from pfeife_amd.hip import HipKernels

    hip = HipKernels(0)
    dy, x = rnd((rows, d), BF16, 1).cuda(), rnd((rows, d), F32, 2).cuda()
    gamma, mean, rstd = rnd((d,), F32, 4).cuda(), torch.zeros(rows, device="cuda"), torch.ones(rows, device="cuda")
    nb, res = hip.norm_bwd_partials(rows), []
    for off in (0, 1, 2, 3):
        dx, lp = torch.zeros(rows, d, device="cuda"), torch.zeros(rows, d, dtype=BF16, device="cuda")
        ws = torch.zeros(nb * 3 * d + 4, device="cuda")[off:off + nb * 3 * d]
        hip.norm_bwd_fused(dy, x, gamma, mean, rstd, None, dx, lp, ws, rows, d, True, True)(torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        res.append((dx.cpu(), ws.view(nb, 3, d).double().sum(0).cpu()))
    bound = rows * 2.0 ** -24 * torch.stack([(dy.double() * x.double()).abs().sum(0), dy.double().abs().sum(0)]).cpu()
    for dx, sums in res[1:]:
        torch.testing.assert_close(dx, res[0][0], rtol=2e-5, atol=8e-5)
        assert bool(((sums - res[0][1])[:2].abs() <= bound + 1e-6).all())
        assert float((sums - res[0][1])[2].abs().max()) <= 2.0 ** -7 * float(res[0][0].abs().sum(0).max())   # (a rounding the other way)
