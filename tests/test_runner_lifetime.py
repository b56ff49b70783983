"""A runner that is dropped goes away with its buffers and its micro-batches' threads (kernel table double on the CPU)."""
import gc
import threading
import weakref

import pytest
import torch
import torch.nn as nn

from oracle.kernels_oracle import OracleKernels
from pfeife_amd.mp import net_states
from pfeife_amd.option import PipeOption


class Model(nn.Module):
    def __init__(self):
        super().__init__()
        self.a, self.b = nn.Linear(8, 8), nn.Linear(8, 8)

    def forward(self, x):
        return self.b(self.a(x))


def runner_after_steps(fail, release):
    from pfeife_amd.mp import PartialRunner, initialize_pfeife, partial_compiler

    torch._dynamo.reset()
    net_states._reset_state_for_tests()
    initialize_pfeife(device="cpu")
    compiled = torch.compile(Model(), backend=partial_compiler)
    runner = PartialRunner(PipeOption(device_cnt=2, batch_cnt=3, batch_size=2, split_points=["b"], mixed_precision=None,
                                      optimizer=dict(type="sgd", lr=0.1)), kernels=OracleKernels("cpu"))
    state = dict(fail=False)

    def fn(x):
        loss = compiled(x).square().mean()
        if state["fail"] and float(x[0, 0]) == 1.0:
            raise ValueError("no loss")
        loss.backward()
        return loss.detach()

    runner.set_exec_fn(fn)
    x = torch.randn(6, 8)
    x[2, 0] = 1.0                  # (the second micro-batch)
    runner.step(x)
    if fail:
        state["fail"] = True
        with pytest.raises(ValueError):
            runner.step(x)
        state["fail"] = False
    for _ in range(2):
        runner.step(x)
    arena = weakref.ref(runner.worker.params._arena)      # what the gradients lie in
    if release:
        runner.worker.release()
    return weakref.ref(runner), arena, runner._batch_threads


@pytest.mark.parametrize("fail", [False, True])
@pytest.mark.parametrize("release", [False, True])
def test_a_dropped_runner_leaves_nothing(fail, release):
    before = threading.active_count()
    runner, arena, threads = runner_after_steps(fail, release)
    assert len(threads) == 3 and all(t.daemon for t in threads)
    # the next runner takes the place of the last one; the compiled graphs are dropped with it
    other = runner_after_steps(False, True)
    gc.collect()
    assert runner() is None and arena() is None
    for t in threads:
        t.join(10)
        assert not t.is_alive()
    assert threading.active_count() <= before + len(other[2])


def test_a_dropped_runner_gives_its_baton_back(monkeypatch):
    from pfeife_amd import hip

    lib, gone = hip.load(), []
    destroy = lib.pf_baton_destroy
    monkeypatch.setattr(lib, "pf_baton_destroy", lambda h: (gone.append(h), destroy(h))[1])
    threads = [runner_after_steps(False, False)[2] for _ in range(3)]
    gc.collect()
    for t in threads[0] + threads[1]:
        t.join(10)
    assert len(set(gone)) >= 2        # (the last runner still is the compiled models')
