"""The fused Adam step against torch's own optimizer, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cls,decay", [(torch.optim.Adam, 0.0), (torch.optim.Adam, 0.1), (torch.optim.AdamW, 0.0), (torch.optim.AdamW, 0.1)])
def test_steps_are_torchs(hip, cls, decay):
    """Sizes with and without remainders of four and of a chunk; gradients from 1e-6 to 1e2, some exactly zero and some that
    cancel the first moment."""
    g = torch.Generator().manual_seed(3)
    ref = [torch.nn.Parameter(torch.randn(n, generator=g).cuda()) for n in (1, 4, 1023, 4099, 100_000)]
    opt = cls(ref, lr=1e-3, weight_decay=decay)
    ours = [[p.detach().clone() for p in ref], *([torch.zeros_like(p.data) for p in ref] for _ in range(3))]
    table, n, chunks = hip.adam_table(*ours)
    s = torch.cuda.current_stream().cuda_stream
    for step in range(1, 6):
        for p, mine in zip(ref, ours[1]):
            grad = (torch.randn(p.numel(), generator=g) * 10.0 ** torch.randint(-6, 3, (p.numel(),), generator=g)).cuda()
            grad[::7] = 0.0
            if step > 1:
                grad[::5] = -opt.state[p]["exp_avg"][::5] * 9.0      # (0.9 m + 0.1 g is rounding alone)
            p.grad = grad
            mine.copy_(grad)
        opt.step()
        hip.adam_step(table, n, chunks, 1e-3, 0.9, 0.999, 1e-8, decay, step, cls is torch.optim.AdamW, s)
        torch.cuda.synchronize()
        for i, p in enumerate(ref):
            st = opt.state[p]
            for mine, theirs in ((ours[2][i], st["exp_avg"]), (ours[3][i], st["exp_avg_sq"]), (ours[0][i], p.detach())):
                assert torch.equal(mine, theirs), (step, i, (mine - theirs).abs().max())
