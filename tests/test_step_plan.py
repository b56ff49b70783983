"""Which jobs of a captured step are one graph (without a GPU)."""
from types import SimpleNamespace

import pytest

from pfeife_amd.mp.step_plan import SMALL_DW, StepPlan


def launches(*names, flops=0.0):
    return [SimpleNamespace(name=n, flops=flops) for n in names]


class Stream:
    def __init__(self, name):
        self.cuda_stream = name


class Recorder:
    """Issuer and kernel table: a graph is the list of its launches' names."""

    def __init__(self):
        self.destroyed = []

    def event(self):
        return "event"

    def destroy_event(self, event):
        pass

    def jobs(self, jobs):
        return jobs

    def capture(self, ls, stream):
        return [l.name for l in ls]

    def destroy_graph(self, graph):
        self.destroyed.append(graph)


def make(jobs_per_stage, dw_flops, lanes):
    """Two stages, two micro-batches, in one job per stage or two."""
    rec = Recorder()
    streams = {k: Stream(k) for k in ("main", (0, True), (0, False), (1, True))}
    nodes = {s: SimpleNamespace(idx=s, rank=s, input_source=[None if s == 0 else (0, 0)]) for s in (0, 1)}
    w = SimpleNamespace(issuer=rec, kernels=rec, part_graph=SimpleNamespace(nodes=nodes, outputs=[(1, 0)]), stream_obj=streams["main"],
                        stream=lambda: 0, lane_mode="rankdir", lanes=None, stack_dw=True, begin_graph=["begin"], mbs={0: None, 1: None},
                        begin_launches=lambda: launches("begin"))
    if lanes:
        w.lanes = {(0, True): streams[0, True], (0, False): streams[0, False], (1, True): streams[1, True], (1, False): streams["main"]}
    w._lane_key = lambda s, f: (s, f)
    w.order = [(s, m, f) for m in (0, 1) for s, f in ((0, True), (1, True))] + [(s, m, False) for m in (0, 1) for s in (1, 0)]
    w.last_forward = {1: 0, 3: 1}
    w.last_backward = {0: 1, 1: 1}
    w.jobs = {}
    for s in (0, 1):
        for mbs in ([[0, 1]] if jobs_per_stage == 1 else [[0], [1]]):
            prog = SimpleNamespace(fwd=launches("f%d" % s), bwd=launches("b%d" % s), fwd_graph=["f%d" % s], bwd_graph=["b%d" % s])
            for m in mbs:
                w.jobs[s, m] = SimpleNamespace(prog=prog, mbs=mbs, first=mbs[0], last=mbs[-1])
    w.dw_jobs = {s: [launches("dw%d" % s, flops=dw_flops / 2), ["dw%d" % s]] for s in (0, 1)}
    return StepPlan(w), rec


def graphs(jobs):
    return [g for g, *_ in jobs if g is not None]


@pytest.mark.parametrize("lanes", [False, True])
def test_jobs_over_all_micro_batches_are_one_graph_each_way(lanes):
    plan, rec = make(1, SMALL_DW, lanes)
    assert graphs(plan._begin) == [["begin", "f0", "f1"]]
    assert [graphs(a) + graphs(b) for (a, b), _ in plan.turns] == [[], []]
    assert graphs(plan._end) == [["b1", "dw1", "b0", "dw0"]]
    assert all(s == "main" and not waits for _, s, waits, _ in plan._begin + plan._end)
    plan.release()
    assert rec.destroyed == [["begin", "f0", "f1"], ["b1", "dw1", "b0", "dw0"]]


@pytest.mark.parametrize("lanes", [False, True])
def test_large_weight_gradients_stay_beside_the_next_stage(lanes):
    plan, _ = make(1, 2 * SMALL_DW, lanes)
    assert graphs(plan._begin) == [["begin", "f0", "f1"]]
    assert graphs(plan._end) == [["b1"], ["dw1"], ["b0"], ["dw0"]]
    by = {tuple(g): (s, waits) for g, s, waits, _ in plan._end if g is not None}
    assert by[("b0",)] == (((0, False), ["event"]) if lanes else ("main", []))      # after b1, not after dw1
    if lanes:
        assert plan._end[-1][:2] == (None, "main") and plan._end[-1][2] == ["event"]    # what follows the step waits for the other lane


@pytest.mark.parametrize("lanes", [False, True])
def test_jobs_per_micro_batch_stay_apart(lanes):
    plan, rec = make(2, 0.0, lanes)
    assert graphs(plan._begin) == [["begin"]]
    assert [g for (a, b), _ in plan.turns for g in graphs(a) + graphs(b)] + graphs(plan._end) == \
        [["f0"], ["f1"], ["f0"], ["f1"], ["b1"], ["b0"], ["b1"], ["dw1"], ["b0"], ["dw0"]]
    plan.release()
    assert rec.destroyed == []
