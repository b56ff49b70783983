"""Products of two tensors, act(a) * b in all its forms: those that run give PyTorch's losses and weights, the others are refused (kernel
table double on the CPU)."""
import copy

import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

from oracle.kernels_oracle import OracleKernels
from pfeife_amd.mp import net_states
from pfeife_amd.option import PipeOption

FORMS = {
    "silu b": lambda a, b, x: F.silu(a(x)) * b(x),
    "a gelu": lambda a, b, x: a(x) * F.gelu(b(x)),
    "silu gelu": lambda a, b, x: F.silu(a(x)) * F.gelu(b(x)),
    "gelu silu": lambda a, b, x: F.gelu(a(x), approximate="tanh") * F.silu(b(x)),
    "silu silu": lambda a, b, x: F.silu(a(x)) * F.silu(b(x)),
    "relu silu": lambda a, b, x: F.relu(a(x)) * F.silu(b(x)),
    "silu of gelu": lambda a, b, x: F.silu(F.gelu(a(x))) * F.gelu(b(x)),
}


class Block(nn.Module):
    def __init__(self, product, bias, dim=32, ffn=40):
        super().__init__()
        self.product = product
        self.inp = nn.Linear(dim, dim)
        self.a, self.b = nn.Linear(dim, ffn, bias=bias), nn.Linear(dim, ffn, bias=bias)
        self.down = nn.Linear(ffn, dim)

    def forward(self, x):
        x = self.inp(x)
        return x + self.down(self.product(self.a, self.b, x))


def steps(product, bias, mixed, n=2):
    from pfeife_amd.mp import PartialRunner, initialize_pfeife, partial_compiler

    torch._dynamo.reset()
    net_states._reset_state_for_tests()
    initialize_pfeife(device="cpu")
    torch.manual_seed(0)
    model = Block(product, bias)
    ref = copy.deepcopy(model)
    runner = PartialRunner(PipeOption(device_cnt=2, batch_cnt=2, batch_size=2, split_points=["down"], mixed_precision=mixed,
                                      optimizer=dict(type="sgd", lr=0.1)), kernels=OracleKernels("cpu"))
    compiled = torch.compile(model, backend=partial_compiler)

    def fn(x):
        loss = compiled(x).float().square().mean()
        loss.backward()
        return loss.detach()

    runner.set_exec_fn(fn)
    x = torch.randn(4, 10, 32, generator=torch.Generator().manual_seed(1)) * 3
    got = torch.cat([torch.stack([l.detach().float() for l in runner.step(x)]) for _ in range(n)])
    want = []
    for _ in range(n):
        ref.zero_grad()
        for i in (0, 2):
            loss = ref(x[i:i + 2]).square().mean()
            loss.backward()
            want.append(loss.detach())
        with torch.no_grad():
            for p in ref.parameters():
                p -= 0.1 * p.grad
    return model, ref, got, torch.stack(want)


@pytest.mark.parametrize("mixed", [None, "bf16"])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("form", FORMS)
def test_is_pytorchs(form, bias, mixed):
    model, ref, got, want = steps(FORMS[form], bias, mixed)
    # bf16: a handful of rounded operands (2^-9 each) in a mean over 640 squares; a missing activation moves the losses by 5 % and more
    torch.testing.assert_close(got, want, rtol=2.0 ** -7 if mixed else 1e-5, atol=0)
    # what the weights moved by: sums of products of such operands in every layer
    torch.manual_seed(0)
    for (name, p), q, r in zip(model.named_parameters(), ref.parameters(), Block(FORMS[form], bias).parameters()):
        assert (p - q).norm() <= (2.0 ** -5 if mixed else 1e-5) * (q - r).norm(), name


def square(a, b, x):
    h = F.silu(a(x))
    return h * h * F.silu(b(x))


@pytest.mark.parametrize("mixed", [None, "bf16"])
@pytest.mark.parametrize("product", [square, lambda a, b, x: F.relu(a(x)) * b(x)], ids=["h * h", "relu b"])
def test_is_refused(product, mixed):
    with pytest.raises(Exception, match="outside the gated-MLP pattern"):
        steps(product, False, mixed, 1)
