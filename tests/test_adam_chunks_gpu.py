"""The Adam step in one pass over memory, against the step that finds its own place."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from pfeife_amd.hip import HipKernels
    return HipKernels()


@pytest.mark.parametrize("sizes", [[1], [1024], [1025, 0, 0, 4], [0, 3, 1023] + [2] * 61 + [0], [5] * 64 + [1_000_003] + [1] * 4100, [0] * 70 + [9]])
def test_one_pass_equals_the_step_that_finds_its_place(hip, sizes):
    """Items before and after 64, 64 * 64 and empty ones, chunks that end inside four elements: bit for bit, scaled and not."""
    def state():
        g = torch.Generator().manual_seed(1)
        return [[(torch.randn(n, generator=g) if j < 3 else torch.rand(n, generator=g)).cuda() for n in sizes] for j in range(4)]

    lib, s = hip.lib, torch.cuda.current_stream().cuda_stream
    hyper = (1e-3, 0.9, 0.999, 1e-8, 0.01)
    for scaled in (False, True):
        a, b = state(), state()
        scaler = [torch.tensor([2.0, 0.0, 0.0, 6.0, 0.0, 0.0, 0.0, 0.0], device="cuda") for _ in range(2)]
        table, n, chunks = hip.adam_table(*a)
        items = torch.tensor([[t.data_ptr() for t in ts] + [ts[0].numel()] for ts in zip(*b)], dtype=torch.int64).cuda()
        if scaled:
            hip.adam_step_scaled(table, n, chunks, *hyper, False, scaler[0], s)
            rc = lib.pf_adam_step_scaled(items.data_ptr(), n, max(sizes), *hyper, 0, scaler[1].data_ptr(), s)
        else:
            hip.adam_step(table, n, chunks, *hyper, 7, False, s)
            rc = lib.pf_adam_step(items.data_ptr(), n, max(sizes), *hyper, 7, 0, s)
        assert rc == 0
        torch.cuda.synchronize()
        for x, y, before in zip(a, b, state()):
            for u, v in zip(x, y):
                assert torch.equal(u, v)
        assert any(not torch.equal(u, v) for u, v in zip(a[0], state()[0]))
