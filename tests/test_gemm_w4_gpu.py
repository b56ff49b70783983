"""The four-wavefront 256x256 tile of the direct-to-LDS kernel (variant 18) at its edges, against the kernel oracle and,
bit for bit, against the eight-wavefront tile (variant 7), which adds up in the same order."""
import pytest
import torch

from test_kernels_gpu import BF16, F16, F32, TOL, close, rnd

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from pfeife_amd.hip import HipKernels

    return HipKernels(0)


@pytest.fixture(scope="module")
def oracle():
    from oracle.kernels_oracle import OracleKernels

    return OracleKernels("cpu")


def _run(hip, oracle, tensors, outs, variant_name, **kw):
    cpu = {k: (None if v is None else v.clone()) for k, v in tensors.items()}
    got = {}
    for variant in (7, 18):
        dev = {k: (None if v is None else v.cuda()) for k, v in tensors.items()}
        launch = hip.gemm(**dev, variant=variant, **kw)
        if variant == 18:
            assert launch.variant.endswith(variant_name), launch.variant
        launch(torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        got[variant] = {o: dev[o].cpu() for o in outs}
    oracle.gemm(**cpu, **kw)()
    for o in outs:
        assert torch.equal(got[7][o], got[18][o]), o
    return {o: (got[18][o], cpu[o]) for o in outs}


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("M,N,K", [(256, 256, 64), (1, 8, 128), (257, 264, 192), (511, 520, 320), (300, 1160, 2048)])
def test_row_major_classes(hip, oracle, dtype, M, N, K):
    """One, two, three stages and more; one tile, ragged tiles, tiles with one row or eight columns."""
    x, w, bias = rnd((M, K), dtype, 1), rnd((N, K), dtype, 2, 0.1), rnd((N,), dtype, 3)
    rt, at = TOL[dtype]
    z16 = lambda: torch.zeros(M, N, dtype=dtype)
    base = dict(M=M, N=N, K=K, lda=K, ldb=K, ldc=N)
    cls = lambda ec: "256, 256, 64, 2, 2, 1, 2, false, false, %d>" % ec
    close(_run(hip, oracle, dict(a=x, b=w, c=z16(), bias=bias), ["c"], cls(0), round_mid=1, **base)["c"], rt, at)
    close(_run(hip, oracle, dict(a=x, b=w, c=torch.zeros(M, N, dtype=F32), bias=bias), ["c"], cls(1), **base)["c"], 1e-3, 1e-2)
    r = _run(hip, oracle, dict(a=x, b=w, c=z16(), bias=bias, aux_out=z16()), ["c", "aux_out"], cls(2), round_mid=1, act=1,
             ld_aux_out=N, **base)
    close(r["c"], rt, at)
    close(r["aux_out"], rt, at)
    close(_run(hip, oracle, dict(a=x, b=w, c=torch.zeros(M, N, dtype=F32), bias=bias, residual=rnd((M, N), F32, 4)), ["c"], cls(3),
               round_mid=1, ld_res=N, **base)["c"], rt, at)
    close(_run(hip, oracle, dict(a=x, b=w, c=z16(), aux_in=rnd((M, N), dtype, 6)), ["c"], cls(5), dact=1, ld_aux_in=N, **base)["c"],
          rt, at * 4)
    close(_run(hip, oracle, dict(a=x, b=w, c=rnd((M, N), dtype, 7)), ["c"], cls(6), beta=1, **base)["c"], rt, at * 2)
    close(_run(hip, oracle, dict(a=x, b=w, c=z16(), bias=bias, residual=rnd((M, N + 8), dtype, 8)), ["c"], cls(7), round_mid=1,
               ld_res=N + 8, **base)["c"], rt, at * 2)


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("M,N,K", [(256, 256, 64), (264, 520, 72), (304, 256, 1021), (512, 8, 200)])
def test_weight_gradients(hip, oracle, dtype, M, N, K):
    """Both operands reduction-strided; depths that are no multiple of a stage."""
    a, b = rnd((K, M), dtype, 1), rnd((K, N), dtype, 2)
    for beta, ec in ((0, 1), (1, 4)):
        r = _run(hip, oracle, dict(a=a, b=b, c=rnd((M, N), F32, 3)), ["c"], "true, true, %d>" % ec, M=M, N=N, K=K, lda=M, ldb=N,
                 ldc=N, a_trans=1, b_trans=1, beta=beta)
        close(r["c"], 1e-4, 2e-3)


@pytest.mark.parametrize("dtype", [F16, BF16])
def test_grouped_weight_gradients(hip, dtype):
    """Products of different sizes, depths and betas in one launch: what each gives alone on the eight-wavefront tile."""
    outs = {}
    for variant in (7, 18):
        members, outs[variant] = [], []
        for i, (M, N, K, beta) in enumerate([(512, 264, 200, 0), (256, 520, 64, 1), (264, 256, 1021, 0)]):
            a, b, c = rnd((K, M + 8), dtype, i).cuda(), rnd((K, N + 16), dtype, i + 3).cuda(), rnd((M, N + 8), F32, i + 6).cuda()
            members.append(hip.gemm(a, b, c, M=M, N=N, K=K, lda=M + 8, ldb=N + 16, ldc=N + 8, a_trans=1, b_trans=1, beta=beta,
                                    variant=variant))
            outs[variant].append(c)
        stream = torch.cuda.current_stream().cuda_stream
        if variant == 18:
            group = hip.gemm_group(members)
            assert group.variant == "gemm16x_group_kernel<%d, 256, 256, 64, 2, 2, 1, 2, true, true, 4>" % (1 if dtype == F16 else 2)
            group(stream)
        else:
            for m in members:
                m(stream)
        torch.cuda.synchronize()
    for x, y in zip(outs[7], outs[18]):
        assert torch.equal(x, y)


def test_column_sums(hip):
    """GELU' with the column sums of what is stored, as partial rows: equal to sums over the stored values."""
    M, N, K = 700, 520, 128
    dy, w, h = rnd((M, K), BF16, 1).cuda(), rnd((N, K), BF16, 2, 0.1).cuda(), rnd((M, N), BF16, 3).cuda()
    c = torch.zeros(M, N, dtype=BF16, device="cuda")
    launch = hip.gemm(dy, w, c, M=M, N=N, K=K, lda=K, ldb=K, ldc=N, dact=1, aux_in=h, ld_aux_in=N, variant=18)
    ws, _, nb, _ = hip.gemm_attach_colsum(launch, lambda shape, dtype: torch.full(shape, float("nan"), dtype=dtype, device="cuda"))
    launch(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    want = c.double().sum(0)
    # (fp32 sums of at most 256 values each)
    assert nb == 3 and float((ws.double().sum(0) - want).abs().max()) <= 256 * 2.0 ** -24 * float(c.double().abs().sum(0).max())


def test_automatic_choice(hip):
    """Long rows and large weight gradients take the tile; depths that are no multiple of 64 and small outputs do not."""
    def name(M, N, K, t=0):
        a = torch.empty(K if t else M, M if t else K, dtype=BF16, device="cuda")
        b = torch.empty(K if t else N, N if t else K, dtype=BF16, device="cuda")
        c = torch.empty(M, N, dtype=F32 if t else BF16, device="cuda")
        return hip.gemm(a, b, c, M=M, N=N, K=K, lda=a.shape[1], ldb=b.shape[1], ldc=N, a_trans=t, b_trans=t).variant

    w4 = "256, 256, 64, 2, 2, 1, 2"
    assert w4 in name(8192, 2048, 2048) and w4 in name(12608, 1024, 4096) and w4 in name(4096, 4096, 12608, 1)
    assert w4 not in name(8192, 2048, 2048 + 32) and w4 not in name(788, 384, 1536) and w4 not in name(2048, 2048, 8192, 1)


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("M,N,K", [(12336, 1408, 256), (6000, 3072, 192), (8200, 4096, 128), (20001, 1024, 128)])
def test_products_in_two_launches(hip, dtype, M, N, K):
    """Rows past the last whole round of large tiles go to a launch of their own: the bits of one launch, for every operand
    that has a row of its own, with row strides wider than N; the column sums to fp32 sums in another order."""
    x, w, bias = rnd((M, K), dtype, 1).cuda(), rnd((N, K), dtype, 2, 0.1).cuda(), rnd((N,), dtype, 3).cuda()
    s = torch.cuda.current_stream().cuda_stream
    wide = lambda dt, seed: rnd((M, N + 8), dt, seed).cuda()
    for kind in ("store", "act", "res32", "acc16", "dact"):
        got = []
        for variant in (0, 9):
            c = wide(F32 if kind == "res32" else dtype, 4)
            aux, ws = wide(dtype, 5), None
            kw = dict(M=M, N=N, K=K, lda=K, ldb=K, ldc=N + 8, round_mid=1, variant=variant)
            if kind == "act":
                kw.update(act=1, aux_out=aux, ld_aux_out=N + 8)
            elif kind == "dact":
                kw.update(dact=1, aux_in=aux, ld_aux_in=N + 8)
            elif kind == "res32":
                kw.update(residual=wide(F32, 6), ld_res=N + 8)
            elif kind == "acc16":
                kw.update(beta=1)
            launch = hip.gemm(x, w, c, bias=None if kind in ("dact", "acc16") else bias, **kw)
            if kind == "dact":
                ws = hip.gemm_attach_colsum(launch, lambda shape, dt: torch.full(shape, float("nan"), dtype=dt, device="cuda"))[0]
            launch(s)
            torch.cuda.synchronize()
            got.append((c, aux, ws))
        (c0, a0, w0), (c1, a1, w1) = got
        assert torch.equal(c0, c1) and torch.equal(a0, a1), kind
        if w0 is not None:
            want = c0[:, :N].double().sum(0)
            assert float((w0.double().sum(0) - want).abs().max()) <= 256 * 2.0 ** -24 * float(c0[:, :N].double().abs().sum(0).max())


@pytest.mark.parametrize("M,N,K", [(12214, 1536, 384), (12922, 1536, 1024), (4728, 4096, 512)])
def test_column_sums_of_two_launches(hip, M, N, K):
    """Two launches of tiles of different heights: as many partial rows as announced, stored values as without them; a workspace for the
    first tile's height alone gets rows of that height.  (Bound: fp32 sums of at most 256 values each.)"""
    dy, w, h = rnd((M, K), BF16, 1).cuda(), rnd((N, K), BF16, 2, 0.1).cuda(), rnd((M, N), BF16, 3).cuda()
    c = [torch.zeros(M, N, dtype=BF16, device="cuda") for _ in range(3)]
    kw = dict(M=M, N=N, K=K, lda=K, ldb=K, ldc=N, dact=1, aux_in=h, ld_aux_in=N)
    s = torch.cuda.current_stream().cuda_stream
    hip.gemm(dy, w, c[0], **kw)(s)
    any_height, one_height = hip.gemm(dy, w, c[1], **kw), hip.gemm(dy, w, c[2], **kw)
    got = []

    def alloc(shape, dtype):
        got.append(torch.full((shape[0] * shape[1] + 64,), float("nan"), dtype=dtype, device="cuda"))
        return got[-1][:shape[0] * shape[1]].view(shape)

    _, _, nb, _ = hip.gemm_attach_colsum(any_height, alloc)
    low = (M + 255) // 256
    assert nb > low and "256, 256, 64, 2, 2" in any_height.variant
    whole = torch.full((low * N + 64,), float("nan"), device="cuda")
    one_height.desc.colsum_ws = whole.data_ptr()
    any_height(s)
    one_height(s)
    torch.cuda.synchronize()
    assert torch.equal(c[0], c[1]) and torch.equal(c[0], c[2])
    want = c[0].double().sum(0)
    for ws, rows in ((got[0], nb), (whole, low)):
        assert ws[rows * N:].isnan().all()
        err = (ws[:rows * N].view(rows, N).double().sum(0) - want).abs().max()
        assert float(err) <= 256 * 2.0 ** -24 * float(c[0].double().abs().sum(0).max())
