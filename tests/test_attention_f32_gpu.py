"""The fp32 attention kernels against 64 bits: column blocks, stages and head dimensions at their edges."""
import copy
import gc

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from pfeife_amd.hip import HipKernels
    return HipKernels()


def exact(q, k, v, d_o, scale, causal):
    """Output and gradients in 64 bits, and what each is a sum of in magnitudes."""
    q, k, v, d_o = (t.double() for t in (q, k, v, d_o))
    s = q @ k.transpose(2, 3).contiguous() * scale
    if causal:
        s = s.masked_fill(torch.ones(s.shape[2:], dtype=torch.bool, device=s.device).triu(1 + s.shape[3] - s.shape[2]), -torch.inf)
    p = s.softmax(-1)
    o, dp = p @ v, d_o @ v.transpose(2, 3).contiguous()
    ds = p * (dp - (d_o * o).sum(-1, keepdim=True)) * scale
    t = lambda x: x.transpose(2, 3).contiguous()
    # roundings: scores (as a factor of p), dP and delta
    e = q.abs() @ t(k.abs()) * scale + 1
    pe = p * e
    dpe = d_o.abs() @ t(v.abs()) + (d_o.abs() * (p @ v.abs())).sum(-1, keepdim=True)
    room = pe * dpe * scale + p * (pe * dpe).sum(-1, keepdim=True) * scale
    return ((o, pe @ v.abs() + p @ v.abs() * pe.sum(-1, keepdim=True)), (ds @ k, room @ k.abs()), (t(ds) @ q, t(room) @ q.abs()),
            (t(p) @ d_o, t(pe) @ d_o.abs() + t(p * pe.sum(-1, keepdim=True)) @ d_o.abs()))


@pytest.mark.parametrize("B,H,Tq,Tk,hd,causal", [
    (1, 1, 1, 1, 4, 0), (2, 3, 5, 5, 16, 1), (1, 2, 15, 33, 20, 0), (2, 1, 64, 64, 32, 1), (1, 2, 65, 31, 36, 0), (4, 6, 197, 197, 64, 0),
    (1, 3, 127, 129, 60, 1), (2, 2, 130, 200, 72, 1), (1, 2, 96, 97, 96, 1), (1, 1, 257, 255, 100, 0), (2, 1, 190, 190, 128, 1),
    (1, 1, 1, 300, 64, 1), (1, 2, 333, 1, 48, 0), (1, 1, 1030, 1030, 64, 1)])
def test_fp32_attention(hip, B, H, Tq, Tk, hd, causal):
    """Queries, keys and values packed per token, gradients into a packed tensor of that layout, and nothing beside them.  Bound: units of
    roundoff of what the sums hold in magnitudes, as many as the longest chain of sums is long."""
    g = torch.Generator().manual_seed(hd + Tk)
    scale = hd ** -0.5
    T = max(Tq, Tk)
    base = torch.randn(B, T, 3, H, hd, generator=g).cuda()
    d_o = torch.randn(B, Tq, H, hd, generator=g).cuda().permute(0, 2, 1, 3)
    heads = lambda t: (t[:, :Tq, 0].permute(0, 2, 1, 3), t[:, :Tk, 1].permute(0, 2, 1, 3), t[:, :Tk, 2].permute(0, 2, 1, 3))
    q, k, v = heads(base)
    dbase, want_rest = torch.full_like(base, 7.0), torch.full_like(base, 7.0)
    o = torch.zeros(B, Tq, H, hd, device="cuda").permute(0, 2, 1, 3)
    lse, delta = torch.zeros(B, H, 2 * Tq, device="cuda"), torch.zeros(B, H, Tq, device="cuda")
    dq, dk, dv = heads(dbase)
    hip.run("attention_fwd", q, k, v, o, lse, scale, causal)
    hip.run("attention_bwd", q, k, v, o, d_o, lse, delta, dq, dk, dv, scale, causal)
    torch.cuda.synchronize()
    for got, (want, room), name in zip((o, dq, dk, dv), exact(q, k, v, d_o, scale, causal), ("o", "dq", "dk", "dv")):
        bound = (hd + T + 8) * 2.0 ** -24 * room + 1e-30
        over = ((got.double() - want).abs() / bound).max()
        assert over <= 1, (name, float(over))
    for t in heads(want_rest):
        t.zero_()
    for t in heads(dbase):
        t.zero_()
    assert torch.equal(dbase, want_rest)


def test_fp32_attention_scores_that_are_not_finite(hip):
    """Overflowing scores give NaN rows, as the softmax through memory does; other rows keep their values."""
    q = torch.randn(1, 1, 40, 64, generator=torch.Generator().manual_seed(1)).cuda()
    clean = torch.zeros_like(q)
    lse = torch.zeros(1, 1, 80, device="cuda")
    hip.run("attention_fwd", q, q, q, clean, lse, 0.125, 1)
    bad = q.clone()
    bad[0, 0, 20] = 1e30       # (its own score and those of later rows with it)
    o = torch.zeros_like(q)
    hip.run("attention_fwd", bad, bad, q, o, lse, 0.125, 1)
    torch.cuda.synchronize()
    assert torch.equal(o[0, 0, :20], clean[0, 0, :20]) and o[0, 0, 20].isnan().all()


def test_fp32_attention_refuses(hip):
    """What the kernels cannot read is an error of the entry point, not a launch."""
    t = torch.zeros(1, 2, 8, 66, device="cuda")
    lse = torch.zeros(1, 2, 16, device="cuda")
    for q in (t, t[..., :62], t[..., 1:65], torch.zeros(1, 2, 8, 132, device="cuda")):
        with pytest.raises(RuntimeError):
            hip.run("attention_fwd", q, q, q, q, lse, 0.125, 0)
    q = torch.zeros(1, 2, 8, 64, device="cuda")
    with pytest.raises(RuntimeError):
        hip.run("attention_fwd", q, q, q, q, lse, -1.0, 0)


class Attend(torch.nn.Module):
    def __init__(self, form, dim, heads, hd, scale):
        super().__init__()
        self.form, self.heads, self.hd, self.scale = form, heads, hd, scale
        self.a = torch.nn.Linear(dim, heads * hd * (3 if form == "packed" else 1))
        self.b = torch.nn.Linear(heads * hd, dim)

    def forward(self, x, ctx):
        split = lambda t: t.view(t.shape[0], t.shape[1], self.heads, -1).transpose(1, 2)
        if self.form == "packed":
            q, k, v = (split(t) for t in self.a(x).chunk(3, -1))
        else:            # keys are the values: two gradients into one tensor; queries with them too, or contiguous by heads
            k = v = split(self.a(ctx))
            q = k if self.form == "same" else split(self.a(x)).contiguous()
        o = F.scaled_dot_product_attention(q, k, v, is_causal=self.form == "packed", scale=self.scale)
        return self.b(o.transpose(1, 2).reshape(o.shape[0], o.shape[2], -1))


@pytest.mark.parametrize("form,heads,hd,scale,T,Tc,fused", [
    ("packed", 2, 16, None, 33, 1, True), ("same", 2, 12, 0.5, 9, 40, True), ("cross", 3, 20, None, 70, 19, True), ("cross", 1, 4, None, 1, 1, True),
    ("packed", 2, 6, None, 20, 1, False), ("cross", 1, 132, None, 10, 12, False), ("cross", 2, 16, -0.3, 20, 17, False),
    ("cross", 1, 16, None, 8, 1040, False), ("packed", 2, 64, None, 1040, 1, True)])
def test_fp32_attention_of_a_stage(form, heads, hd, scale, T, Tc, fused):
    """Which calls take the fused kernels, and losses and gradients against 64 bits on either way."""
    from pfeife_amd.mp import PartialRunner, initialize_pfeife, net_states, partial_compiler
    from pfeife_amd.mp.partial.module import PartialModule
    from pfeife_amd.option import PipeOption

    old = PartialModule._runner
    if old is not None and getattr(old, "worker", None) is not None:
        old.worker.release()
        old.exec_fn = None
    PartialModule._runner = None
    torch._dynamo.reset()
    gc.collect()
    net_states._reset_state_for_tests()
    initialize_pfeife()
    torch.manual_seed(0)
    model = Attend(form, 24, heads, hd, scale)
    ref = copy.deepcopy(model).double()
    runner = PartialRunner(PipeOption(device_cnt=2, batch_cnt=2, batch_size=2, split_points=["b"], optimizer=dict(type="sgd", lr=0.0)))
    model.cuda()
    cmodel = torch.compile(model, backend=partial_compiler)

    def fn(x, ctx):
        loss = cmodel(x, ctx).float().square().mean()
        loss.backward()
        return loss.detach()

    runner.set_exec_fn(fn)
    g = torch.Generator().manual_seed(1)
    x, ctx = torch.randn(4, T, 24, generator=g), torch.randn(4, Tc, 24, generator=g)
    want = []
    for i in (0, 2):
        loss = ref(x[i:i + 2].double(), ctx[i:i + 2].double()).square().mean()
        loss.backward()
        want.append(float(loss.detach()))
    for _ in range(3):      # job by job, captured, from job lists
        losses = runner.step(x.cuda(), ctx.cuda())
        torch.cuda.synchronize()
        for got, w in zip(losses, want):
            assert abs(float(got) - w) <= 1e-5 * w
        for (n, p), (_, r) in zip(model.named_parameters(), ref.named_parameters()):
            # (a key's bias gradient is zero but for rounding: sizes are compared over the whole parameter)
            assert (p.grad.cpu().double() - r.grad).abs().max() <= 2e-5 * r.grad.abs().max() + 1e-9, n
    names = {getattr(l, "kernel", "") for slot in runner.worker.mbs.values() for p in slot.stage_programs.values()
             for l in list(p.fwd) + list(p.bwd)}
    assert ({"pf_attention_f32_fwd", "pf_attention_f32_bwd"} <= names) == fused and ("pf_softmax_fwd" in names) == (not fused)
