"""fp32 products by wavefronts that split the depth: every tile at its edges, against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from pfeife_amd.hip import HipKernels
    return HipKernels()


def operand(rows, cols, seed):
    """Rows wider than the operand: what lies behind a row's end must not get into the products."""
    g = torch.Generator().manual_seed(seed)
    t = torch.full((rows, (cols + 3) // 4 * 4 + 4), float("nan"))
    t[:, :cols] = torch.randn(rows, cols, generator=g)
    return t.cuda()


@pytest.mark.parametrize("a_trans,b_trans", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("tile,M,N,K", [("1, 2, 6", 17, 33, 192), ("2, 2, 4", 500, 350, 1000), ("2, 3, 4", 801, 330, 1530),
                                        ("3, 3, 3", 383, 1530, 3151), ("3, 4, 2", 787, 1540, 381), ("4, 4, 2", 2040, 2043, 251),
                                        ("4, 5, 4", 3153, 385, 1535), ("4, 5, 2", 3150, 1537, 383)])
def test_depth_split_tiles(hip, tile, M, N, K, a_trans, b_trans):
    """Stages that end inside a fragment, tiles past the last row and column, stored and accumulated with every operand of the epilogue.
    The bound of a sum of K products in any order: (K + 4) units of roundoff of the sum of magnitudes."""
    a, b = operand(*((K, M) if a_trans else (M, K)), 1), operand(*((K, N) if b_trans else (N, K)), 2)
    am = (a[:, :M].t() if a_trans else a[:, :K]).double().contiguous()
    bm = (b[:, :N] if b_trans else b[:, :K].t()).double().contiguous()
    prod, mags = am @ bm, am.abs() @ bm.abs()
    kw = dict(M=M, N=N, K=K, lda=a.shape[1], ldb=b.shape[1], ldc=N + 3, a_trans=a_trans, b_trans=b_trans)
    s = torch.cuda.current_stream().cuda_stream

    def wide(seed):
        return torch.randn(M, N + 3, generator=torch.Generator().manual_seed(seed)).cuda()

    c = wide(3)
    keep = c.clone()
    launch = hip.gemm(a, b, c, **kw)
    assert launch.variant == "gemm32k_kernel<%s, %s, %s>" % (tile, "true" if a_trans else "false", "true" if b_trans else "false")
    launch(s)
    torch.cuda.synchronize()
    bound = (K + 4) * 2.0 ** -24 * mags
    assert ((c[:, :N].double() - prod).abs() <= bound).all()
    assert torch.equal(c[:, N:], keep[:, N:])          # nothing behind a row's end is written
    c, res, bias = wide(4), wide(5), torch.randn(N, generator=torch.Generator().manual_seed(6)).cuda()
    want = 0.5 * prod + bias.double() + res[:, :N].double() + c[:, :N].double()
    room = 0.5 * bound + 2.0 ** -22 * (0.5 * mags + bias.double().abs() + res[:, :N].double().abs() + c[:, :N].double().abs())
    hip.gemm(a, b, c, bias=bias, residual=res, ld_res=N + 3, beta=1, alpha=0.5, **kw)(s)
    torch.cuda.synchronize()
    assert ((c[:, :N].double() - want).abs() <= room).all()


@pytest.mark.parametrize("b_trans", [0, 1])
def test_depth_split_batches(hip, b_trans):
    """Batches (attention's products over memory at 250 tokens): every entry has operands and results of its own."""
    nb, T, hd = 6, 250, 72
    g = torch.Generator().manual_seed(7)
    p = torch.randn(nb, T, 252, generator=g).cuda()
    v = torch.randn(nb, T if b_trans else hd, 72 if b_trans else 252, generator=g).cuda()
    o = torch.zeros(nb, T, hd).cuda()
    launch = hip.gemm(p, v, o, T, hd, T, 252, v.shape[2], hd, b_trans=b_trans, batch=(2, 3), sa=(3 * T * 252, T * 252),
                      sb=(3 * v.stride(0), v.stride(0)), sc=(3 * T * hd, T * hd))
    assert launch.variant.startswith("gemm32k_kernel")
    launch(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    pd = p[:, :, :T].double().contiguous()
    vd = (v if b_trans else v[:, :, :T].transpose(1, 2)).double().contiguous()
    assert ((o.double() - pd @ vd).abs() <= (T + 4) * 2.0 ** -24 * (pd.abs() @ vd.abs())).all()
