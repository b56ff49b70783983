"""Linear layers that read one input and meet in one attention or gated product run as one product: which do, and that results are those
of the layers one by one (kernel table double on the CPU)."""
import copy
import functools

import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

from oracle.kernels_oracle import OracleKernels
from pfeife_amd.executor import lowering
from pfeife_amd.mp import net_states
from pfeife_amd.option import PipeOption


class Block(nn.Module):
    def __init__(self, form, dim=32, heads=4, hd=8, ctx=24, ffn=40):
        super().__init__()
        bias = form == "bias"
        width = heads * hd if form != "width" else heads * 7
        self.form, self.heads = form, heads
        self.inp = nn.Linear(dim, dim)
        self.q = nn.Linear(dim, width, bias=bias)
        self.k = nn.Linear(ctx if form == "cross" else dim, width, bias=bias)
        self.v = nn.Linear(ctx if form == "cross" else dim, width, bias=bias)
        self.o = nn.Linear(width, dim)
        self.gate = nn.Linear(dim, ffn, bias=False)
        self.up = nn.Linear(dim, ffn, bias=False)
        self.down = nn.Linear(ffn, dim)
        if form == "tied":
            self.v.weight = self.k.weight
        if form == "frozen":
            self.k.weight.requires_grad_(False)

    def forward(self, x, ctx):
        x = self.inp(x)
        c = ctx if self.form == "cross" else x
        h = lambda t: t.view(t.shape[0], t.shape[1], self.heads, -1).transpose(1, 2)
        q, k, v = self.q(x), self.k(c), self.v(c)
        if self.form == "seen":          # the values are read by something else as well
            x = x + v
        o = F.scaled_dot_product_attention(h(q), h(k), h(v), is_causal=self.form == "causal")
        x = x + self.o(o.transpose(1, 2).reshape(x.shape[0], x.shape[1], -1))
        return x + self.down(F.silu(self.gate(x)) * self.up(x))


class Table(OracleKernels):
    @functools.wraps(OracleKernels.gemm)
    def gemm(self, a, b, c, **kw):
        self.seen.append((kw["N"], kw["K"]))
        return super().gemm(a, b, c, **kw)


def step(form, mixed, joint, monkeypatch, steps=2):
    from pfeife_amd.mp import PartialRunner, initialize_pfeife, partial_compiler

    torch._dynamo.reset()
    net_states._reset_state_for_tests()
    initialize_pfeife(device="cpu")
    torch.manual_seed(0)
    model = Block(form)
    ref = copy.deepcopy(model)
    table = Table("cpu")
    table.seen = []
    monkeypatch.undo()
    if not joint:
        monkeypatch.setattr(lowering, "_joint_layers", lambda L, node: None)
    runner = PartialRunner(PipeOption(device_cnt=2, batch_cnt=2, batch_size=2, split_points=["down"], mixed_precision=mixed,
                                      optimizer=dict(type="sgd", lr=0.05)), kernels=table)
    cmodel = torch.compile(model, backend=partial_compiler)

    def fn(x, ctx):
        loss = cmodel(x, ctx).float().square().mean()
        loss.backward()
        return loss.detach()

    runner.set_exec_fn(fn)
    g = torch.Generator().manual_seed(1)
    x, ctx = torch.randn(4, 10, 32, generator=g), torch.randn(4, 6, 24, generator=g)
    # the second step reads the shadows of updated weights
    losses = [torch.stack([l.detach().float() for l in runner.step(x, ctx)]) for _ in range(steps)]
    return model, ref, torch.cat(losses), table.seen, (x, ctx)


# (N, K) of products that only the joint layers have, forward
@pytest.mark.parametrize("form,mixed,joint", [
    ("self", "bf16", [(96, 32), (80, 32)]), ("causal", "fp16", [(96, 32), (80, 32)]), ("cross", "bf16", [(64, 24), (80, 32)]),
    ("frozen", "bf16", [(96, 32), (80, 32)]), ("bias", "bf16", [(80, 32)]), ("seen", "bf16", [(64, 32), (80, 32)]),
    ("width", "bf16", [(80, 32)]), ("tied", "bf16", [(80, 32)]), ("self", None, [])])
def test_layers_of_one_input(form, mixed, joint, monkeypatch):
    model, ref, losses, seen, (x, ctx) = step(form, mixed, True, monkeypatch)
    apart, _, losses1, seen1, _ = step(form, mixed, False, monkeypatch)
    assert not set(seen1) & {(96, 32), (80, 32), (64, 24), (64, 32)}
    assert set(seen) & {(96, 32), (80, 32), (64, 24), (64, 32)} == set(joint)
    # the same but for 16-bit sums after every layer's input gradient
    tol = {"bf16": 2.0 ** -7, "fp16": 2.0 ** -10, None: 0.0}[mixed]
    torch.testing.assert_close(losses, losses1, rtol=tol, atol=0)
    for (n, p), (_, q) in zip(model.named_parameters(), apart.named_parameters()):
        assert (p - q).norm() <= tol * q.norm(), n
        assert (p.grad is None) == (q.grad is None)
        if p.grad is not None and n != "k.bias":      # (a key bias moves all scores of a row alike: its gradient is rounding alone)
            assert (p.grad - q.grad).norm() <= 4 * tol * q.grad.norm(), n
    # and against autograd in fp32
    for i in (0, 2):
        ref(x[i:i + 2], ctx[i:i + 2]).square().mean().backward()
    with torch.no_grad():
        for p in ref.parameters():
            if p.grad is not None:
                p -= 0.05 * p.grad
    for (n, p), (_, q) in zip(model.named_parameters(), ref.named_parameters()):
        assert (p.grad is None) == (q.grad is None), n
    want = torch.stack([ref(x[i:i + 2], ctx[i:i + 2]).square().mean().detach() for i in (0, 2)])
    torch.testing.assert_close(losses[2:], want, rtol=max(4 * tol, 1e-5), atol=0)
