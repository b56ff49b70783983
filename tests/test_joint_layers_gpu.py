"""Linear layers that run as one product, on the device: whole steps against those of the layers one by one and against autograd in fp32."""
import functools

import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

from pfeife_amd.option import PipeOption

pytestmark = pytest.mark.gpu


class Block(nn.Module):
    def __init__(self, form, dim=64, heads=4, hd=24, ctx=40, ffn=88):
        super().__init__()
        self.form, self.heads = form, heads
        cross = ctx if form == "cross" else dim
        self.inp = nn.Linear(dim, dim)
        self.q, self.k, self.v = (nn.Linear(d, heads * hd, bias=False) for d in (dim, cross, cross))
        self.gate, self.up = nn.Linear(dim, ffn, bias=False), nn.Linear(dim, ffn, bias=False)
        self.o, self.down = nn.Linear(heads * hd, dim), nn.Linear(ffn, dim)

    def forward(self, x, ctx):
        x = self.inp(x)
        c = ctx if self.form == "cross" else x
        h = lambda t: t.view(t.shape[0], t.shape[1], self.heads, -1).transpose(1, 2)
        o = F.scaled_dot_product_attention(h(self.q(x)), h(self.k(c)), h(self.v(c)), is_causal=self.form == "causal")
        x = x + self.o(o.transpose(1, 2).reshape(x.shape[0], x.shape[1], -1))
        return x + self.down(F.silu(self.gate(x)) * self.up(x))


def gradients(form, mixed, tokens, joint, monkeypatch):
    from pfeife_amd.executor import lowering
    from pfeife_amd.hip import HipKernels
    from pfeife_amd.mp import PartialRunner, initialize_pfeife, partial_compiler
    from pfeife_amd.mp.net_states import _reset_state_for_tests

    torch._dynamo.reset()
    _reset_state_for_tests()
    initialize_pfeife()
    torch.manual_seed(0)
    model = Block(form).cuda()
    seen = []
    with monkeypatch.context() as m:
        gemm = HipKernels.gemm

        @functools.wraps(gemm)
        def seeing(self, a, b, c, **kw):
            seen.append((kw["N"], kw["K"]))
            return gemm(self, a, b, c, **kw)

        m.setattr(HipKernels, "gemm", seeing)
        if not joint:
            m.setattr(lowering, "_joint_layers", lambda L, node: None)
        runner = PartialRunner(PipeOption(device_cnt=2, batch_cnt=2, batch_size=2, split_points=["down"], mixed_precision=mixed, loss_scale=1.0,
                                          optimizer=dict(type="sgd", lr=0.0)))
        compiled = torch.compile(model, backend=partial_compiler)

        def fn(x, ctx):
            loss = compiled(x, ctx).float().square().mean()
            loss.backward()
            return loss.detach()

        runner.set_exec_fn(fn)
        g = torch.Generator().manual_seed(1)
        x, ctx = torch.randn(4, tokens, 64, generator=g).cuda(), torch.randn(4, 9, 40, generator=g).cuda()
        for _ in range(4):               # job by job, then graphs
            losses = torch.stack([l.float() for l in runner.step(x, ctx)])
        torch.cuda.synchronize()
    got = {n: p.grad.clone() for n, p in model.named_parameters()}
    runner.worker.release()
    model.zero_grad()
    want = torch.stack([model(x[i:i + 2], ctx[i:i + 2]).square().mean() for i in (0, 2)])
    want.sum().backward()
    return losses, want.detach(), got, {n: p.grad for n, p in model.named_parameters()}, set(seen)


# tokens: few rows, and 256 rows and more (the input's gradient multiplies by the transposed weights)
@pytest.mark.parametrize("tokens", [5, 149])
@pytest.mark.parametrize("form,mixed", [("self", "bf16"), ("causal", "fp16"), ("cross", "bf16")])
def test_layers_of_one_input(form, mixed, tokens, monkeypatch):
    losses, want, got, exact, seen = gradients(form, mixed, tokens, True, monkeypatch)
    losses1, _, got1, _, seen1 = gradients(form, mixed, tokens, False, monkeypatch)
    own = {(192, 40), (176, 64)} if form == "cross" else {(288, 64), (176, 64)}
    assert own <= seen and not own & seen1
    tol = {"bf16": 2.0 ** -7, "fp16": 2.0 ** -10}[mixed]       # (a handful of operands rounded to half of that each)
    torch.testing.assert_close(losses, losses1, rtol=tol, atol=0)
    torch.testing.assert_close(losses, want, rtol=tol, atol=0)
    for n in exact:
        apart = (got1[n] - exact[n]).norm()
        assert (got[n] - exact[n]).norm() <= 1.25 * apart + tol / 4 * exact[n].norm(), n       # (no further off than the layers apart)
