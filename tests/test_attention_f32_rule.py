"""Which fp32 attention goes to the fused kernels: nothing that their entry points refuse (no GPU: shapes alone)."""
import ctypes
import itertools

import pytest
import torch

from pfeife_amd import hip
from pfeife_amd.executor.lowering import _f32_heads, _fused_f32

PF_ERR_HIP = -3


def heads(B, H, T, hd, between=0, layout="bthd"):
    """[B, H, T, hd] of a layout, `between` elements after every token's row."""
    shape = dict(b=B, h=H, t=T)
    strides, at = {}, hd + between
    for c in reversed(layout[:-1]):
        strides[c] = at
        at *= shape[c]
    return torch.empty_strided((B, H, T, hd), (strides["b"], strides["h"], strides["t"], 1), dtype=torch.float32, device="meta")


def accepted(q, k, v, scale):
    """Whether the entry points take it.  There is no GPU here: what passes their checks fails at the launch."""
    if torch.cuda.is_available():
        pytest.skip("made-up addresses: not where the kernels would run")
    d = hip.AttnDesc()
    d.dtype, d.B, d.H, d.Tq, d.Tk, d.hd, d.scale = hip.PF_F32, q.shape[0], q.shape[1], q.shape[2], k.shape[2], q.shape[3], scale
    o = torch.empty((q.shape[0], q.shape[2], q.shape[1], q.shape[3]), device="meta").permute(0, 2, 1, 3)
    for name, t in dict(q=q, k=k, v=v, o=o, d_o=o, dq=q, dk=k, dv=v).items():
        setattr(d, name, 1 << 20)
        prefix = "do" if name == "d_o" else name
        for axis, s in zip("bht", t.stride()[:3]):
            setattr(d, "%s_s%s" % (prefix, axis), s)
    d.lse = d.delta = 1 << 20
    lib = hip.load()
    return all(fn(ctypes.byref(d), None) == PF_ERR_HIP for fn in (lib.pf_attention_f32_fwd, lib.pf_attention_f32_bwd))


def test_what_the_rule_takes_the_kernels_take():
    taken = 0
    sizes = [(1, 1, 16, 16, 16), (2, 3, 5, 77, 64), (4, 8, 1024, 1024, 128), (1, 1, 64, 4096, 64), (1, 128, 16, 16 * 65535, 8), (1, 128, 16, 16 * 65535 + 1, 8),
             (1, 128, 16 * 65535 + 1, 16, 8), (1 << 12, 1 << 11, 16, 16, 4), (1 << 12, (1 << 11) - 1, 16, 16, 4), (8192, 8, 32, 32, 128), (8191, 8, 32, 32, 128),
             (1, 1 << 17, 16, 16, 64), (1, (1 << 17) - 1, 16, 16, 64), (2, 2, 40, 40, 6)]
    for (B, H, Tq, Tk, hd), between, layout, scale in itertools.product(sizes, (0, 2, 4, (1 << 23) - 16), ("bthd", "bhtd", "tbhd"), (0.125, 0.0, -1.0)):
        q, k, v = heads(B, H, Tq, hd, between, layout), heads(B, H, Tk, hd, between, layout), heads(B, H, Tk, hd, between, layout)
        if not _fused_f32(q, k, v, scale):
            continue
        taken += 1
        assert accepted(q, k, v, scale), (B, H, Tq, Tk, hd, between, layout)
    assert taken > 30
    assert _f32_heads(heads(8191, 8, 32, 128, layout="tbhd")) and not _f32_heads(heads(8192, 8, 32, 128, layout="tbhd"))
