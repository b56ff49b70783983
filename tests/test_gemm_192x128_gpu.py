"""The 192x128 tile (variant 19) at its edges, every epilogue class of row-major products, against the kernel oracle and, bit for
bit, against the eight-wavefront 256x256 tile (variant 7), which adds up in the same order; and where the choice takes it."""
import pytest
import torch

from test_gemm_w4_gpu import hip, oracle  # noqa: F401  (fixtures)
from test_kernels_gpu import BF16, F16, F32, TOL, close, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("M,N,K", [(192, 128, 64), (1, 8, 128), (193, 136, 192), (575, 264, 320), (400, 1160, 1024)])
def test_row_major_classes(hip, oracle, dtype, M, N, K):  # noqa: F811
    x, w, bias = rnd((M, K), dtype, 1), rnd((N, K), dtype, 2, 0.1), rnd((N,), dtype, 3)
    rt, at = TOL[dtype]
    z16, base = torch.zeros(M, N, dtype=dtype), dict(M=M, N=N, K=K, lda=K, ldb=K, ldc=N)
    for ec, tensors, kw, tol in (
            (0, dict(c=z16, bias=bias), dict(round_mid=1), (rt, at)),
            (1, dict(c=torch.zeros(M, N), bias=bias), {}, (1e-3, 1e-2)),
            (2, dict(c=z16, bias=bias, aux_out=z16.clone()), dict(round_mid=1, act=1, ld_aux_out=N), (rt, at)),
            (3, dict(c=torch.zeros(M, N), bias=bias, residual=rnd((M, N), F32, 4)), dict(round_mid=1, ld_res=N), (rt, at)),
            (5, dict(c=z16, aux_in=rnd((M, N), dtype, 6)), dict(dact=1, ld_aux_in=N), (rt, at * 4)),
            (6, dict(c=rnd((M, N), dtype, 7)), dict(beta=1), (rt, at * 2)),
            (7, dict(c=z16, bias=bias, residual=rnd((M, N + 8), dtype, 8)), dict(round_mid=1, ld_res=N + 8), (rt, at * 2))):
        tensors, got = dict(tensors, a=x, b=w), {}
        for variant in (7, 19):
            dev = {k: v.clone().cuda() for k, v in tensors.items()}
            launch = hip.gemm(**dev, variant=variant, **kw, **base)
            if variant == 19:
                assert launch.variant.endswith("192, 128, 64, 4, 2, 1, 3, false, false, %d>" % ec), launch.variant
            launch(torch.cuda.current_stream().cuda_stream)
            torch.cuda.synchronize()
            got[variant] = dev
        cpu = {k: v.clone() for k, v in tensors.items()}
        oracle.gemm(**cpu, **kw, **base)()
        for out in ("c", "aux_out"):
            if out in tensors:
                assert torch.equal(got[7][out], got[19][out]), (ec, out)
                close((got[19][out].cpu(), cpu[out]), *tol)


def test_column_sums(hip):  # noqa: F811
    """GELU' leaves one partial row of column sums per 192 rows."""
    M, N, K = 500, 264, 128
    dy, w, h = rnd((M, K), BF16, 1).cuda(), rnd((N, K), BF16, 2, 0.1).cuda(), rnd((M, N), BF16, 3).cuda()
    c = torch.zeros(M, N, dtype=BF16, device="cuda")
    launch = hip.gemm(dy, w, c, M=M, N=N, K=K, lda=K, ldb=K, ldc=N, dact=1, aux_in=h, ld_aux_in=N, variant=19)
    ws, _, nb, _ = hip.gemm_attach_colsum(launch, lambda shape, dtype: torch.full(shape, float("nan"), dtype=dtype, device="cuda"))
    launch(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    want = c.double().sum(0)
    # (fp32 sums of at most 192 values each)
    assert nb == 3 and float((ws.double().sum(0) - want).abs().max()) <= 192 * 2.0 ** -24 * float(c.double().abs().sum(0).max())


def test_automatic_choice(hip):  # noqa: F811
    """Outputs that it covers in one round and 256x128 in a round with a third of the device idle; depths that are no
    multiple of 64, several rounds and reduction-strided products do not take it."""
    def name(M, N, K, t=0):
        a = torch.empty(K if t else M, M if t else K, dtype=F16, device="cuda")
        b = torch.empty(K if t else N, N if t else K, dtype=F16, device="cuda")
        c = torch.empty(M, N, dtype=F32 if t else F16, device="cuda")
        return hip.gemm(a, b, c, M=M, N=N, K=K, lda=a.shape[1], ldb=b.shape[1], ldc=N, a_trans=t, b_trans=t).variant

    tile = "192, 128, 64, 4, 2, 1, 3"
    assert tile in name(4096, 1280, 1280) and tile in name(4096, 1280, 5120) and tile in name(3072, 1408, 1408)
    assert tile not in name(4096, 1280, 1280 + 32) and tile not in name(8192, 1280, 1280) and tile not in name(4096, 1280, 5120, 1)
