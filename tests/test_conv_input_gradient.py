"""3x3 and 1x1 "same" convolutions: the input gradient as one product with the taps in reverse (kernel table double on the CPU)."""
import copy
import functools

import pytest
import torch
import torch.nn as nn

from oracle.kernels_oracle import OracleKernels
from pfeife_amd.mp import net_states
from pfeife_amd.option import PipeOption


class Convs(nn.Module):
    def __init__(self, a, b, c, k):
        super().__init__()
        self.c0 = nn.Conv2d(a, b, 1)
        self.c1 = nn.Conv2d(b, c, k, padding=k // 2)
        self.c2 = nn.Conv2d(c, b, 3, padding=1, bias=False)

    def forward(self, x):
        x = self.c0(x)
        return x + self.c2(self.c1(x))          # the first gradient is added to, the others stored


@pytest.mark.parametrize("mixed", [None, "bf16"])
@pytest.mark.parametrize("channels,k,H,W,wide", [((8, 16, 24), 3, 13, 11, True), ((8, 8, 16), 1, 20, 9, True), ((8, 16, 24), 3, 5, 3, False),
                                                 ((4, 12, 20), 3, 13, 11, None)])
def test_input_gradients(channels, k, H, W, wide, mixed):
    """Against autograd in fp32.  wide: 256 pixels and more in a micro-batch and channels of whole 16 bytes, the condition of the one product
    (None: in fp32 alone)."""
    from pfeife_amd.mp import PartialRunner, initialize_pfeife, partial_compiler

    if mixed and wide is None:
        pytest.skip("16-bit products need channels in eights")
    calls = []

    class Table(OracleKernels):
        def im2col3x3(self, src, dst, B, H, W, C, flip=0):
            calls.append(flip)
            return super().im2col3x3(src, dst, B, H, W, C, flip)

    torch._dynamo.reset()
    net_states._reset_state_for_tests()
    initialize_pfeife(device="cpu")
    torch.manual_seed(0)
    model = Convs(*channels, k)
    ref = copy.deepcopy(model)
    runner = PartialRunner(PipeOption(device_cnt=2, batch_cnt=2, batch_size=2, split_points=["c2"], mixed_precision=mixed,
                                      optimizer=dict(type="sgd", lr=0.0)), kernels=Table("cpu"))
    cmodel = torch.compile(model, backend=partial_compiler)

    def fn(x):
        loss = cmodel(x).float().square().mean()
        loss.backward()
        return loss.detach()

    runner.set_exec_fn(fn)
    x = torch.randn(4, channels[0], H, W, generator=torch.Generator().manual_seed(1))
    for _ in range(2):
        losses = runner.step(x)
        want = []
        ref.zero_grad()
        for i in (0, 2):
            loss = ref(x[i:i + 2]).square().mean()
            loss.backward()
            want.append(float(loss.detach()))
        tol = 1e-5 if mixed is None else 2e-2
        for a, b in zip(losses, want):
            assert abs(float(a) - b) <= tol * b
        for (n, p), (_, q) in zip(model.named_parameters(), ref.named_parameters()):
            assert (p.grad - q.grad).norm() <= tol * q.grad.norm(), n
    one = wide or wide is None
    assert (1 in calls) == one and (0 in calls) == (wide is not None or mixed is None)


class Wider(nn.Module):
    def __init__(self, c=16, o=48):
        super().__init__()
        self.c0, self.c1, self.c2 = nn.Conv2d(8, c, 1), nn.Conv2d(c, o, 3, padding=1), nn.Conv2d(o, 8, 1)

    def forward(self, x):
        return self.c2(self.c1(self.c0(x)))


def wider_steps(mixed, channels, monkeypatch, check):
    """Two steps' gradients against autograd in fp32; -> (N, K) of the products."""
    from pfeife_amd.mp import PartialRunner, initialize_pfeife, partial_compiler

    gemm, calls = OracleKernels.gemm, []

    @functools.wraps(gemm)
    def seen(self, a, b, c, **kw):
        check(kw)
        calls.append((kw["N"], kw["K"]))
        return gemm(self, a, b, c, **kw)

    monkeypatch.setattr(OracleKernels, "gemm", seen)
    torch._dynamo.reset()
    net_states._reset_state_for_tests()
    initialize_pfeife(device="cpu")
    torch.manual_seed(0)
    model = Wider(*channels)
    ref = copy.deepcopy(model)
    runner = PartialRunner(PipeOption(device_cnt=2, batch_cnt=2, batch_size=2, split_points=["c2"], mixed_precision=mixed,
                                      optimizer=dict(type="sgd", lr=0.0)), kernels=OracleKernels("cpu"))
    cmodel = torch.compile(model, backend=partial_compiler)

    def fn(x):
        loss = cmodel(x).float().square().mean()
        loss.backward()
        return loss.detach()

    runner.set_exec_fn(fn)
    x = torch.randn(4, 8, 13, 11, generator=torch.Generator().manual_seed(1))
    for _ in range(2):
        runner.step(x)
        ref.zero_grad()
        for i in (0, 2):
            ref(x[i:i + 2]).square().mean().backward()
        for (n, p), (_, q) in zip(model.named_parameters(), ref.named_parameters()):
            assert (p.grad - q.grad).norm() <= (2e-2 if mixed else 1e-5) * q.grad.norm(), n      # (as above)
    return calls


@pytest.mark.parametrize("limit,one", [(300_000, False), (600_000, True)])
def test_windows_of_the_gradient_fit_an_operand(limit, one, monkeypatch):
    """More channels out than in: the forward windows may fit the size a 16-bit operand can have and the gradient's may not, which then takes the
    product with the windows as its result.  The limit is lowered, and held to as pf_gemm holds to it."""
    from pfeife_amd.executor import lowering, merge

    monkeypatch.setattr(lowering, "MAX_BYTES", limit)
    monkeypatch.setattr(merge, "MAX_BYTES", limit)

    def check(kw):
        for rows, ld in ((kw["K"] if kw.get("a_trans") else kw["M"], kw["lda"]), (kw["K"] if kw.get("b_trans") else kw["N"], kw["ldb"])):
            assert (rows + 256) * ld * 2 < limit

    calls = wider_steps("bf16", (16, 48), monkeypatch, check)
    assert ((16, 9 * 48) in calls) == one and ((9 * 16, 48) in calls) != one


@pytest.mark.parametrize("mixed", [None, "bf16"])
@pytest.mark.parametrize("channels,one", [((8, 768), True), ((8, 776), False), ((200, 776), True)])
def test_many_channels_out_of_few_keep_the_product_of_windows(channels, one, mixed, monkeypatch):
    c, o = channels
    calls = wider_steps(mixed, channels, monkeypatch, lambda kw: None)
    assert ((c, 9 * o) in calls) == one and ((9 * c, o) in calls) != one


def test_the_form_of_the_input_gradient():
    from pfeife_amd.executor.lowering import _windows_of_gradient as one

    assert one(1 << 15, 320, 960, 4) and not one(1 << 15, 320, 968, 4)                       # three times as many at any size
    assert one(20_000, 128, 512, 2) and not one(22_000, 128, 512, 2) and not one(22_000, 64, 512, 2)    # eight times: up to 200 MB
    assert one(9_000, 300, 1200, 2) and not one(9_000, 299, 1200, 2) and not one(10_000, 300, 1200, 2)                        # ... above 768 of them four times
    assert one(5_000, 8, 768, 2) and not one(6_000, 8, 768, 2)                               # others: up to 80 MB
    assert one(100_000, 640, 640, 2) and not one(196_608, 320, 640, 2) and one(196_608, 320, 640, 4)   # 2 GiB of 16 bits
