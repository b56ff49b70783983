"""Layers of one input whose results pass through views: as one product only where every view is one of a range of columns as well
and a gated product gets matrices; otherwise they run apart, as any layer does (kernel table double on the CPU)."""
import functools

import pytest
import torch
import torch.nn.functional as F

from oracle.kernels_oracle import OracleKernels
from pfeife_amd.executor import lowering

from test_gated_product import steps

FFN = 40      # of both layers, over 32 columns


def gated(form):
    def product(a, b, x):
        shape = x.shape[:-1] + (FFN,)
        return (F.silu(form(a(x))) * form(b(x))).view(shape)
    return product


def attention(q_form, k_form, back):
    def product(a, b, x):
        q, k = q_form(a(x)), k_form(b(x))
        return back(F.scaled_dot_product_attention(q, k, k)).reshape(x.shape[:-1] + (FFN,))
    return product


heads = lambda t: t.view(2, 10, 5, 8).transpose(1, 2)
tokens = lambda t: t.transpose(1, 2)
GATED = {
    "plain": (lambda t: t, True), "rows": (lambda t: t.view(20, FFN), True), "rows by reshape": (lambda t: t.reshape(-1, FFN), True),
    "and back": (lambda t: t.view(20, 5, 8).view(2, 10, FFN), True),
    "flat": (lambda t: t.view(-1), False), "flat by reshape": (lambda t: t.reshape(-1), False),
    "heads below each other": (lambda t: t.view(2 * 10 * 5, 8), False), "heads as tokens": (lambda t: t.view(2, 50, 8), False),
    "heads": (lambda t: t.view(2, 10, 5, 8), False), "pairs of tokens": (lambda t: t.view(2, 5, 2 * FFN), False),
}
ATTENTION = {
    "heads": (heads, heads, tokens, True),
    "heads by permute": (lambda t: t.view(20, 5, 8).view(2, 10, 5, 8).permute(0, 2, 1, 3), heads, tokens, True),
    # (apart as well such a reshape copies)
    "one batch": (lambda t: heads(t).reshape(1, 10, 10, 8), lambda t: heads(t).reshape(1, 10, 10, 8), lambda t: t.reshape(2, 5, 10, 8).transpose(1, 2), True),
    "heads as tokens": (lambda t: t.view(2, 50, 1, 8).transpose(1, 2), lambda t: t.view(2, 50, 1, 8).transpose(1, 2), tokens, False),
    "queries flat": (lambda t: t.view(2, 1, 50, 8), lambda t: t.view(2, 1, 50, 8), lambda t: t, False),
}
PRODUCTS = {"gated, " + n: (gated(f), j) for n, (f, j) in GATED.items()}
PRODUCTS.update({"attention, " + n: (attention(q, k, b), j) for n, (q, k, b, j) in ATTENTION.items()})


@pytest.mark.parametrize("form", PRODUCTS)
def test_joint_where_the_views_allow_it(form, monkeypatch):
    product, joint = PRODUCTS[form]
    seen = []
    gemm = OracleKernels.gemm

    @functools.wraps(gemm)
    def seeing(self, a, b, c, **kw):
        seen.append((kw["N"], kw["K"]))
        return gemm(self, a, b, c, **kw)

    monkeypatch.setattr(OracleKernels, "gemm", seeing)
    model, ref, got, want = steps(product, False, "bf16")
    assert ((2 * FFN, 32) in seen) == joint
    torch.testing.assert_close(got, want, rtol=2.0 ** -7, atol=0)      # (a handful of operands rounded to 2^-9 each)
    # the layers one by one: the same but for 16-bit sums after every layer's input gradient
    monkeypatch.setattr(lowering, "_joint_layers", lambda L, node: None)
    apart, _, got1, _ = steps(product, False, "bf16")
    torch.testing.assert_close(got, got1, rtol=2.0 ** -7 if joint else 0, atol=0)
    for (name, p), q in zip(model.named_parameters(), apart.parameters()):
        assert (p - q).norm() <= (2.0 ** -7 if joint else 0) * q.norm(), name
