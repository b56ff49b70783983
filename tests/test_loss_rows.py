"""Cross entropy over all but the last positions of each sequence: the rows are read where they lie and the gradient of the whole
is written at once.  Which slices do so, and that losses and gradients are torch's (kernel table double on the CPU; kernels on the GPU)."""
import copy
import functools

import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

from oracle.kernels_oracle import OracleKernels
from pfeife_amd.mp import net_states
from pfeife_amd.option import PipeOption

V = 24


class Head(nn.Module):
    def __init__(self, form):
        super().__init__()
        self.form = form
        self.body, self.head = nn.Linear(16, 16), nn.Linear(16, V)

    def forward(self, x, y):
        z = self.head(F.gelu(self.body(x)))
        f = self.form
        if f in ("last", "float", "ignored"):
            rows, lab = z[:, :-1, :].reshape(-1, V), y[:, 1:]
        elif f in ("last3", "twice", "seen", "other"):
            rows, lab = z[:, :-3].reshape(-1, V), y[:, 3:]
        elif f == "first":
            rows, lab = z[:, 1:].reshape(-1, V), y[:, 1:]
        elif f == "step":
            rows, lab = z[:, ::2].reshape(-1, V), y[:, ::2]
        elif f == "classes":
            rows, lab = z[:, :-1, :16].reshape(-1, 16), y[:, 1:]
        elif f == "batch":
            rows, lab = z[:-1].reshape(-1, V), y[1:]
        loss = F.cross_entropy(rows.float() if f == "float" else rows, lab.reshape(-1))
        if f == "twice":     # two losses on overlapping regions of one product
            loss = loss + F.cross_entropy(z[:, :-1].reshape(-1, V), y[:, 1:].reshape(-1))
        if f == "seen":      # the whole has a gradient of its own
            loss = loss + F.cross_entropy(z.reshape(-1, V), y.reshape(-1))
        if f == "other":     # the rows have another reader
            loss = loss + F.cross_entropy(F.gelu(rows), lab.reshape(-1))
        return loss


class Table(OracleKernels):
    @functools.wraps(OracleKernels.cross_entropy_fwd)
    def cross_entropy_fwd(self, *a, **kw):
        self.gaps.append(a[8:] if len(a) > 8 else (kw.get("group", 0), kw.get("gap", 0)))
        return super().cross_entropy_fwd(*a, **kw)


@pytest.mark.parametrize("mixed", [None, "bf16"])
@pytest.mark.parametrize("form,gaps", [("last", [(6, 1)]), ("float", [(6, 1)]), ("ignored", [(6, 1)]), ("last3", [(4, 3)]),
                                       ("twice", [(4, 3), (6, 1)]), ("seen", [(4, 3), (0, 0)]), ("other", [(0, 0)]), ("first", [(0, 0)]),
                                       ("step", [(0, 0)]), ("classes", [(0, 0)]), ("batch", [(0, 0)])])
def test_rows_in_place(form, gaps, mixed):
    from pfeife_amd.mp import PartialRunner, initialize_pfeife, partial_compiler

    torch._dynamo.reset()
    net_states._reset_state_for_tests()
    initialize_pfeife(device="cpu")
    torch.manual_seed(0)
    model = Head(form)
    ref = copy.deepcopy(model)
    table = Table("cpu")
    table.gaps = []
    runner = PartialRunner(PipeOption(device_cnt=1, batch_cnt=2, batch_size=3, split_points=None, mixed_precision=mixed,
                                      optimizer=dict(type="sgd", lr=0.0)), kernels=table)
    cmodel = torch.compile(model, backend=partial_compiler)

    def fn(x, y):
        loss = cmodel(x, y)
        loss.backward()
        return loss.detach()

    runner.set_exec_fn(fn)
    g = torch.Generator().manual_seed(1)
    x, y = torch.randn(6, 7, 16, generator=g), torch.randint(0, V, (6, 7), generator=g)
    if form == "classes":
        y %= 16
    if form == "ignored":
        y[0, 2:] = -100
    for _ in range(2):
        for p in model.parameters():
            p.grad = None
        losses = runner.step(x, y)
    want = []
    for xb, yb in zip(x.chunk(2), y.chunk(2)):
        loss = ref(xb, yb)
        loss.backward()
        want.append(loss.detach())
    assert set(table.gaps) == set(gaps)
    # 16-bit activations through two layers: 2^-8 an operand
    tol = 2e-5 if mixed is None else 2e-2
    torch.testing.assert_close(torch.stack([l.float() for l in losses]), torch.stack(want), rtol=tol, atol=tol)
    for p, r in zip(model.parameters(), ref.parameters()):
        torch.testing.assert_close(p.grad, r.grad, rtol=tol, atol=tol * r.grad.abs().max().item())


@pytest.mark.gpu
@pytest.mark.parametrize("out", ["same", "fp16"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("groups,group,gap,classes,shift", [(1, 5, 1, 40, 0), (3, 7, 1, 24, 0), (2, 6, 3, 2056, 0), (4, 1, 1, 8, 0),
                                                           (3, 4, 2, 37, 0), (2, 3, 1, 32, 1), (2, 5, 0, 48, 0)])
def test_gap_kernels(groups, group, gap, classes, shift, dtype, out):
    from pfeife_amd import hip

    k = hip.HipKernels()
    g = torch.Generator("cuda").manual_seed(3)
    n, rows = groups * (group + gap) * classes, groups * group
    logits = (torch.randn(n + shift, device="cuda", generator=g) * 3).to(dtype)[shift:]
    targets = torch.randint(0, classes, (rows,), device="cuda", generator=g)
    if rows > 3:
        targets[1] = -100
    row_loss, row_lse, loss = (torch.empty(m, device="cuda") for m in (rows, rows, 2))
    k.run("cross_entropy_fwd", logits, targets, row_loss, row_lse, loss, rows, classes, -100, group, gap)
    ref = logits.double().view(groups, group + gap, classes).requires_grad_()
    want = F.cross_entropy(ref[:, :group].reshape(-1, classes), targets)
    want.backward()
    odt = dtype if out == "same" else torch.float16
    dl = torch.full((n + shift,), float("nan"), device="cuda", dtype=odt)[shift:]
    k.run("cross_entropy_bwd", logits, targets, row_lse, torch.ones(1, device="cuda"), loss, dl, rows, classes, -100, group, gap)
    torch.cuda.synchronize()
    torch.testing.assert_close(loss[0].double(), want.detach(), rtol=1e-5, atol=1e-5)
    got = dl.view(groups, group + gap, classes)
    assert (got[:, group:] == 0).all()
    # exp(x - lse) with |x - lse| below 32: 32 * 2^-23 of fp32's argument, and half a unit of the result's type
    rel = 2.0 ** -18 + {torch.float32: 0.0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[odt]
    torch.testing.assert_close(got.double(), ref.grad, rtol=rel, atol=2.0 ** -24)
