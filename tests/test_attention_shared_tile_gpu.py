"""Attention over 257 to 288 tokens: the ninth tile of 32, which a workgroup's eight wavefronts share (the queries of
the forward and of dQ, the keys of dK / dV), one row of it to all, beside long, short and one-token other axes (their
operands in LDS are then smaller than the partial results), with and without a causal mask (rows that see no key of a
wavefront's share), against the kernel oracle and torch's attention."""
import pytest
import torch

import test_kernels_gpu as base
from test_gemm_w4_gpu import hip, oracle  # noqa: F401  (fixtures)
from test_kernels_gpu import BF16, F16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("Tq,Tk,hd,causal", [
    (257, 257, 64, 0), (288, 288, 96, 0), (257, 288, 88, 1), (288, 257, 32, 0), (258, 1, 88, 0), (1, 258, 96, 0),
    (270, 40, 64, 0), (33, 270, 40, 1), (271, 271, 80, 1), (129, 160, 96, 0), (256, 256, 72, 1)])
def test_ninth_tile(hip, oracle, dtype, Tq, Tk, hd, causal):  # noqa: F811
    base.test_fused_attention(hip, oracle, dtype, dict(B=2, H=3, Tq=Tq, Tk=Tk, hd=hd, causal=causal, packed=False))
