"""Stage jobs over several micro-batches (pfeife_amd/executor/merge.py) on the kernel oracle: a step whose jobs are
merged against the same step with one job per micro-batch."""
import copy

import pytest
import torch
import torch.nn.functional as F

from pfeife_amd.bench_models.llama import LlamaConfig, LlamaForCausalLM
from pfeife_amd.bench_models.unet_stage import UNetStage, UNetStageConfig
from pfeife_amd.bench_models.vit import ViTConfig, VisionTransformer
from pfeife_amd.executor.merge import MicroBatchLayout
from pfeife_amd.option import PipeOption
from test_host_pipeline import make_runner


def _model(family):
    torch.manual_seed(0)
    if family == "vit":
        return VisionTransformer(ViTConfig(image_size=32, patch_size=16, dim=64, depth=2, heads=2, mlp_dim=128, num_classes=16))
    if family == "decoder":
        return LlamaForCausalLM(LlamaConfig(vocab=64, dim=64, layers=2, heads=2, ffn=88, max_seq=9))
    return UNetStage(UNetStageConfig(in_channels=32, channels=64, temb_dim=32, context_dim=24, heads=2, layers=1))


def _gpu_runner(option):
    from pfeife_amd.mp import PartialRunner, initialize_pfeife, net_states

    torch._dynamo.reset()
    net_states._reset_state_for_tests()
    initialize_pfeife()
    return PartialRunner(option)


def _steps(family, mixed, batch, micro, rows, steps, monkeypatch, device="cpu"):
    """[(results, gradients)] of some steps, and the worker.  `batch`: samples of each step."""
    from pfeife_amd.mp import partial_compiler

    monkeypatch.setenv("PFEIFE_JOB_ROWS", str(rows))
    model = _model(family).to(device)
    make = make_runner if device == "cpu" else _gpu_runner
    splits = {"vit": ["blocks.1"], "decoder": ["layers.1"], "unet": None}[family]
    runner = make(PipeOption(device_cnt=2 if splits else 1, batch_cnt=micro, batch_size=1, split_points=splits,
                                    mixed_precision=mixed, optimizer=dict(type="sgd", lr=0.01)))
    cmodel = torch.compile(model, backend=partial_compiler, dynamic=False)

    def fn(*a):
        if family == "vit":
            loss = F.cross_entropy(cmodel(a[0]).float(), a[1])
        elif family == "decoder":
            loss = cmodel(a[0], a[0])
        else:
            loss = F.mse_loss(cmodel(*a[:3]).float(), a[3])
        loss.backward()
        return loss.detach()

    runner.set_exec_fn(fn)
    out = []
    for n in (batch if isinstance(batch, tuple) else (batch,) * steps):
        g = torch.Generator().manual_seed(n)
        if family == "vit":
            args = (torch.randn(n, 3, 32, 32, generator=g), torch.randint(0, 10, (n,), generator=g))
        elif family == "decoder":
            args = (torch.randint(0, 64, (n, 9), generator=g),)
        else:
            args = (torch.randn(n, 32, 6, 6, generator=g), torch.randn(n, 32, generator=g),
                    torch.randn(n, 5, 24, generator=g), torch.randn(n, 64, 6, 6, generator=g))
        losses = [float(l) for l in runner.step(*(a.to(device) for a in args))]
        out.append((losses, {k: p.grad.cpu().clone() for k, p in model.named_parameters()}))
    return out, runner.worker


@pytest.mark.parametrize("mixed", [None, "bf16"])
@pytest.mark.parametrize("family,batch,micro,rows,jobs", [
    ("vit", 8, 4, 10 ** 6, [[0, 1, 2, 3]]), ("vit", 8, 4, 20, [[0, 1], [2, 3]]), ("vit", 10, 5, 25, [[0, 1, 2], [3, 4]]),
    ("vit", 7, 3, 10 ** 6, [[0, 1, 2]]), ("vit", 3, 3, 10 ** 6, [[0, 1, 2]]), ("vit", 11, 4, 27, [[0, 1], [2, 3]]),
    ("vit", (8, 8, 10, 8, 7), 4, 10 ** 6, None),
    ("decoder", 4, 4, 10 ** 6, [[0, 1, 2, 3]]), ("decoder", 5, 3, 10 ** 6, [[0, 1], [2]]),    # (the last: a loss of one sample)
    ("unet", 4, 2, 10 ** 6, [[0, 1]]), ("unet", 3, 2, 10 ** 6, [[0], [1]]),    # (its channel bias sums sample by sample: other lists)
])
def test_merged_jobs_equal_jobs_per_micro_batch(monkeypatch, family, batch, micro, rows, jobs, mixed):
    """Losses bit for bit (every row is computed from the same operands by the same arithmetic); gradients to the
    rounding of fp32 sums in another order: at most 144 rows (four images of 36 pixels), 144 * 2^-24 = 8.6e-6; in
    16 bits, after an update, to what it changes in the weights' rounding."""
    want, w0 = _steps(family, mixed, batch, micro, 0, 2, monkeypatch)
    got, w = _steps(family, mixed, batch, micro, rows, 2, monkeypatch)
    assert all(len(j.mbs) == 1 for j in w0.jobs.values())
    if jobs is not None:
        assert [sorted(j.mbs) for (s, m), j in sorted(w.jobs.items()) if s == 0 and m == j.mbs[0]] == jobs
        assert all(j.first == min(j.mbs) and j.last == max(j.mbs) for j in w.jobs.values())
    tol = 8.6e-6 if mixed is None else 2e-2
    for i, ((l0, g0), (l1, g1)) in enumerate(zip(want, got)):
        assert all(abs(a - b) <= (0 if i == 0 and mixed else tol * abs(a)) for a, b in zip(l0, l1)), (i, l0, l1)
        for k in g0:
            d = float((g0[k].double() - g1[k].double()).norm() / (g0[k].double().norm() + 1e-30))
            assert d <= tol, (i, k, d)


@pytest.mark.gpu
@pytest.mark.parametrize("mixed", [None, "bf16"])
@pytest.mark.parametrize("family,batch,micro,rows", [
    ("vit", 8, 4, 10 ** 6), ("vit", 8, 4, 20), ("vit", 7, 3, 10 ** 6), ("vit", (8, 8, 8, 10, 8, 8, 7), 4, 10 ** 6),
    ("decoder", 5, 5, 10 ** 6), ("decoder", 5, 3, 10 ** 6), ("unet", 4, 2, 10 ** 6)])
def test_merged_jobs_on_the_device(monkeypatch, family, batch, micro, rows, mixed):
    """Launch by launch, captured and from job lists (four steps): gradients to the rounding of fp32 sums, with 16-bit
    operands to that of a dozen layers (2.5e-2, as every whole-step test here)."""
    if family == "unet" and mixed is None:
        pytest.skip("a stage that runs in 16 bits")
    want, _ = _steps(family, mixed, batch, micro, 0, 4, monkeypatch, "cuda")
    got, w = _steps(family, mixed, batch, micro, rows, 4, monkeypatch, "cuda")
    assert any(len(j.mbs) > 1 for j in w.jobs.values())
    tol = 1e-4 if mixed is None else 2.5e-2
    for i, ((l0, g0), (l1, g1)) in enumerate(zip(want, got)):
        assert all(abs(a - b) <= tol * abs(a) for a, b in zip(l0, l1)), (i, l0, l1)
        for k in g0:
            d = float((g0[k].double() - g1[k].double()).norm() / (g0[k].double().norm() + 1e-30))
            assert d <= tol, (i, k, d)


@pytest.mark.gpu
@pytest.mark.parametrize("family,batch,micro,rows", [("vit", 58, 4, 10 ** 6), ("vit", 59, 4, 140), ("decoder", 26, 3, 10 ** 6)])
def test_merged_ragged_weight_gradients_keep_their_sums(monkeypatch, family, batch, micro, rows):
    """Micro-batches of different sizes, of 64 rows and more each (products of fewer are joined): the first step's matrix
    gradients are those of separate jobs bit for bit."""
    (want,), _ = _steps(family, "bf16", batch, micro, 0, 1, monkeypatch, "cuda")
    (got,), w = _steps(family, "bf16", batch, micro, rows, 1, monkeypatch, "cuda")
    assert any(len(j.mbs) > 1 for j in w.jobs.values())
    # (not the classifier: one row per sample)
    linear = [k for k, g in want[1].items() if g.dim() == 2 and "emb" not in k and "tok" not in k and k != "head.weight"]
    assert want[0] == got[0] and len(linear) >= 4
    for k in linear:
        assert torch.equal(want[1][k], got[1][k]), k


def test_merged_lists_are_as_short_as_one_micro_batchs(monkeypatch):
    """Nothing but a loss inside the model stays per micro-batch."""
    for family, per_mb in (("vit", 0), ("decoder", 2 * 3)):    # cross entropy forward and backward of the last stage
        _, w = _steps(family, "bf16", 8, 4, 10 ** 6, 1, monkeypatch)
        one = sum(len(p.fwd) + len(p.bwd) for p in w.mbs[0].stage_programs.values())
        assert sum(len(p.fwd) + len(p.bwd) for p in w.step_programs()) == one + per_mb


@pytest.mark.parametrize("rows,batch,jobs", [(0, 8, 1), (1, 8, 1), (36, 8, 2), (10 ** 6, 8, 4), (36, 11, 2), (0, 7, 1)])
def test_attention_scratch_is_that_of_one_job(monkeypatch, rows, batch, jobs):
    """Scores, their gradients and the rounded ones (fp32: attention through memory): one buffer for a lane's jobs, with
    room for as many micro-batches as a job takes; nothing is left of the ones it was first lowered with."""
    _, w = _steps("decoder", None, batch, 4, rows, 2, monkeypatch)
    assert {len(j.mbs) for j in w.jobs.values()} == {jobs}
    bufs = {}
    for slot in w.mbs.values():
        for prog in slot.stage_programs.values():
            for l in prog.fwd + prog.bwd:
                for name in {"softmax_fwd": ("s",), "softmax_bwd": ("dp", "ds")}.get(l.call[0] if hasattr(l, "call") else "", ()):
                    bufs.setdefault(name, set()).add(l.call[1][name])
    assert set(bufs) == {"s", "dp", "ds"}
    for name, ts in bufs.items():
        sizes = sorted(t.numel() for t in ts)
        assert len({t.data_ptr() for t in ts}) == (jobs if batch == 8 or jobs > 1 else 2), name   # (two shapes: a buffer each)
        held = {t.untyped_storage().data_ptr(): t.untyped_storage().nbytes() for t in ts}
        assert sum(held.values()) <= 4 * (jobs * sizes[-1] if jobs > 1 or batch == 8 else sum(set(sizes))), name
    kept = {id(t) for ts in bufs.values() for t in ts}
    assert all(id(t) in kept for (_, slot, _, _), t in w.pool._scratch.items() if str(slot).startswith("attn"))


@pytest.mark.parametrize("mixed,products", [("bf16", 4), (None, 1)])
def test_weight_gradients_over_the_step_keep_to_the_operand_limit(monkeypatch, mixed, products):
    """Rows of all micro-batches that make an operand of a 16-bit product larger than pf_gemm takes: a product per
    micro-batch, the same gradients (sums of at most 40 rows in another order, 40 * 2^-24 = 2.4e-6).  fp32 has no such limit."""
    import pfeife_amd.executor.lowering as lowering

    (want,), w0 = _steps("vit", mixed, 8, 4, 0, 1, monkeypatch)
    monkeypatch.setattr(lowering, "MAX_BYTES", (300 * 128) * 2)        # (40 rows in all; qkv has 192 columns)
    (got,), w = _steps("vit", mixed, 8, 4, 0, 1, monkeypatch)
    for worker, n in ((w0, 1), (w, products)):
        job = [l.call[1]["c"].data_ptr() for l in worker.dw_jobs[0][0] if getattr(l, "call", ("",))[0] == "gemm"]
        qkv = [p.grad.data_ptr() for p in worker.params.params if tuple(p.shape) == (192, 64)]
        assert {job.count(c) for c in qkv if c in job} == {n}
    assert want[0] == got[0]
    for k in want[1]:
        assert float((want[1][k] - got[1][k]).norm()) <= 2.4e-5 * float(want[1][k].norm()), k


def test_a_micro_batch_that_differs_keeps_its_own_launches(monkeypatch):
    """Operands that do not follow each other: the launches stay as they are, in order."""
    from oracle.kernels_oracle import OracleKernels
    from pfeife_amd.executor.merge import CallRecorder, Merger

    k = CallRecorder(OracleKernels("cpu"))
    x, y, z = torch.arange(12.0), torch.zeros(12), torch.zeros(12)
    m = Merger(k, torch.empty)
    calls = [k.cast(x[0:4], y[0:4], 4), k.cast(x[4:8], y[4:8], 4), k.cast(x[8:12], z[0:4], 4)]
    out = m.lists([[c] for c in calls])
    assert len(out) == 2 and out[1] is calls[2]
    for l in out:
        l(None)
    assert torch.equal(y[:8], x[:8]) and torch.equal(z[:4], x[8:])
    assert m.lists([[calls[0]], [k.cast(x[4:8], y[6:10], 4)]])[0] is calls[0]      # a gap
    assert m.lists([[calls[0]], [k.fill(y[4:8], 0.0, 4)]])[0] is calls[0]         # another kernel
    assert m.lists([[calls[0]], []]) is None                                       # another structure


def test_shapes_of_a_step_take_one_walk_per_micro_batch(monkeypatch):
    import torch.utils._pytree as pytree
    from pfeife_amd.mp.partial.module import PartialRunner

    walks, steps = [], []
    flatten = pytree.tree_flatten
    runner = make_runner(PipeOption(device_cnt=1, batch_cnt=3, batch_size=1))
    runner.set_exec_fn(lambda *a, **k: None)
    monkeypatch.setattr(PartialRunner, "_probe_forward", lambda self, *a: None)
    monkeypatch.setattr(PartialRunner, "_run_step", lambda self, *a: steps.append((self.worker.uniform_mbs, self.worker.mb_sizes)))
    for args, kwargs, want in [((torch.zeros(8, 2),), dict(y=torch.zeros(8)), (False, [3, 3, 2])),
                               ((torch.zeros(6, 2), torch.zeros(6)), {}, (True, [2, 2, 2]))]:
        runner.step(*args, **kwargs)
        with monkeypatch.context() as m:      # (the split walks too: how often beside that)
            m.setattr(pytree, "tree_flatten", lambda *a, **k: walks.append(1) or flatten(*a, **k))
            from pfeife_amd.batch import split_args_kwargs
            split_args_kwargs(args, kwargs, 3)
            split, walks[:] = len(walks), []
            runner.step(*args, **kwargs)
            assert len(walks) - split == 3
            walks.clear()
        assert steps[-1] == want


@pytest.mark.parametrize("sizes", [[2] * 5, [3, 3, 2, 2], [1, 1, 0, 0], [4]])
@pytest.mark.parametrize("rows", [1, 7, 10 ** 6])
def test_layout_places_do_not_overlap(sizes, rows):
    lay = MicroBatchLayout(sizes, "t")
    lay.form_groups(3, rows)
    assert [m for a, b in lay.groups for m in range(a, b)] == list(range(len(sizes)))
    for in_group in (False, True):
        for per in (1, 6):
            spans = [(m, lay.place(m, in_group).span(per * n)) for m, n in enumerate(sizes) if n]
            for m, (off, total) in spans:
                assert 0 <= off and off + per * sizes[m] <= total == spans[0][1][1]
            for (m, (a, _)), (m2, (b, _)) in zip(spans, spans[1:]):
                if not in_group or lay.group(m) == lay.group(m2):
                    assert b == a + per * sizes[m]


class _TwiceThroughABlock(torch.nn.Module):
    """A stage that uses its weights twice (layers that share parameters)."""

    def __init__(self):
        super().__init__()
        self.up, self.down, self.head = torch.nn.Linear(64, 128), torch.nn.Linear(128, 64), torch.nn.Linear(64, 16)

    def forward(self, x):
        for _ in range(2):
            x = x + self.down(F.gelu(self.up(x)))
        return self.head(x)


def _grouping_kernels():
    """The kernel oracle with the device's way to put weight gradients together: the products of one launch run side by
    side, so each adds to its accumulator as that was before the launch."""
    from types import SimpleNamespace

    from oracle.kernels_oracle import OracleKernels

    class GroupingKernels(OracleKernels):
        GEMM_GROUP_MAX = 8
        groups = []      # every launch of several products, as their accumulators

        def gemm(self, a, b, c, M, N, K, lda, ldb, ldc, a_trans=0, b_trans=0, batch=(1, 1), sa=(0, 0), sb=(0, 0), sc=(0, 0),
                 alpha=1.0, beta=0, bias=None, round_mid=0, aux_out=None, ld_aux_out=0, act=0, dact=0, aux_in=None, ld_aux_in=0,
                 residual=None, ld_res=0, variant=0, unscale_by=None, nonfinite_flag=None):
            launch = super().gemm(a, b, c, M, N, K, lda, ldb, ldc, a_trans, b_trans, batch, sa, sb, sc, alpha, beta, bias, round_mid,
                                  aux_out, ld_aux_out, act, dact, aux_in, ld_aux_in, residual, ld_res, unscale_by, nonfinite_flag)
            launch.desc = SimpleNamespace(M=M, N=N, K=K, C=c.data_ptr(), beta=beta, in_dtype=a.dtype)
            launch.acc = c
            launch.group_key = "tile %d" % variant if a_trans and b_trans and a.dtype != torch.float32 and K >= 64 else ""
            return launch

        @staticmethod
        def gemm_groupable(launch):
            return getattr(launch, "group_key", "") != ""

        def gemm_retiled(self, launch, variant):
            new = lambda stream=None: launch(stream)
            new.desc, new.acc, new.group_key = launch.desc, launch.acc, "tile %d" % variant
            return new

        def gemm_group(self, launches):
            assert 2 <= len(launches) <= self.GEMM_GROUP_MAX and len({l.group_key for l in launches}) == 1
            self.groups.append([l.acc.data_ptr() for l in launches])

            def launch(stream=None):
                before = [l.acc.clone() for l in launches]
                for l, acc in zip(launches, before):
                    l.acc.copy_(acc)
                    l(stream)

            launch.group_key = "group"
            return launch

    return GroupingKernels("cpu")


def _steps_of_shared_weights(monkeypatch, rows, device="cpu"):
    from pfeife_amd.mp import PartialRunner, initialize_pfeife, net_states, partial_compiler

    monkeypatch.setenv("PFEIFE_JOB_ROWS", str(rows))
    torch._dynamo.reset()
    net_states._reset_state_for_tests()
    initialize_pfeife(**(dict(device="cpu") if device == "cpu" else {}))
    torch.manual_seed(0)
    model = _TwiceThroughABlock().to(device)
    kernels = _grouping_kernels() if device == "cpu" else None
    runner = PartialRunner(PipeOption(device_cnt=1, batch_cnt=4, batch_size=1, mixed_precision="bf16", optimizer=dict(type="sgd", lr=0.0)),
                           kernels=kernels)
    cmodel = torch.compile(model, backend=partial_compiler, dynamic=False)

    def fn(x):
        loss = cmodel(x).float().square().mean()
        loss.backward()
        return loss.detach()

    runner.set_exec_fn(fn)
    g = torch.Generator().manual_seed(1)
    for _ in range(4 if device == "cuda" else 1):     # (launch by launch, captured, from job lists)
        runner.step(torch.randn(58, 5, 64, generator=g).to(device))
    return {k: p.grad.cpu().clone() for k, p in model.named_parameters()}, runner.worker, kernels


def _same_shared_gradients(want, got):
    for k in want:
        if want[k].dim() == 2:
            assert torch.equal(want[k], got[k]), k
        assert float((want[k] - got[k]).norm()) <= 1.1e-4 * float(want[k].norm()), k


def test_products_into_one_accumulator_are_never_one_launch(monkeypatch):
    """Weights used twice in a stage, micro-batches of different sizes (15, 15, 14, 14 samples of 5 rows): each accumulator
    gets the products of separate jobs in their order, so that the weights' gradients are the same bit for bit.  (Biases
    add at most 75 rows x 2 uses in another order: 150 * 2^-24 = 9e-6 of the sum of magnitudes, some sqrt(150) times the sum's.)"""
    want, _, _ = _steps_of_shared_weights(monkeypatch, 0)
    got, w, kernels = _steps_of_shared_weights(monkeypatch, 10 ** 6)
    assert any(len(j.mbs) > 1 for j in w.jobs.values()) and kernels.groups
    assert all(len(set(g)) == len(g) for g in kernels.groups), kernels.groups
    _same_shared_gradients(want, got)


@pytest.mark.gpu
def test_weights_used_twice_on_the_device(monkeypatch):
    want, _, _ = _steps_of_shared_weights(monkeypatch, 0, "cuda")
    got, w, _ = _steps_of_shared_weights(monkeypatch, 10 ** 6, "cuda")
    assert any(len(j.mbs) > 1 for j in w.jobs.values())
    _same_shared_gradients(want, got)
