"""The work a program built on this framework has it do: whole optimisation steps through `PartialRunner.step`.

A case is one training program: a model family, its sizes, the precision, the micro-batches of a step and the stage
boundaries.  `prepare` is what such a program holds before a step: the compiled model with its runner, started from the
same checkpoint every time, and one batch on the GPU.  `run` is one `step` on that batch: micro-batch split, forward and
backward of every stage in the schedule's order, loss, gradient accumulation, loss scaling and the Adam step.

A process has one active `PartialRunner` (the compiled graphs find it through the class), so the states of one case
share the program and differ in their batches, as the iterations of a training loop do; preparing another case's state
puts the program of the case before it away.
"""
import gc
import math

import torch
import torch.nn.functional as F

from pfeife_amd.bench_models import llama, unet_stage, vit
from pfeife_amd.loss import CrossEntropyLoss
from pfeife_amd.mp import PartialRunner, initialize_pfeife, partial_compiler
from pfeife_amd.option import PipeOption

LR = 1e-5


def listed():
    return [
        # the smallest step: the two-block classifier of the smoke test, where only launches and host work count
        _vit("vit_tiny_fp32", "fp32", batch=4, micro=2, image=32, patch=16, dim=64, depth=2, heads=4, mlp=128, classes=10,
             splits="blocks.1", ranks=2),
        # a small decoder in four looped stages over two ranks, eight micro-batches: the schedule's longest job list
        _decoder("decoder_looped_bf16", "bf16", batch=16, micro=8, vocab=512, dim=256, depth=4, heads=4, ffn=688, seq=128,
                 splits="layers.1,layers.2,layers.3", ranks=2),
        # ViT-S/16 in full precision, the configuration that also runs on a CPU
        _vit("vit_s16_fp32", "fp32", batch=16, micro=4, image=224, patch=16, dim=384, depth=12, heads=6, mlp=1536,
             classes=1000, splits="blocks.6", ranks=2),
        # fine-tuning ViT-S/16 with a batch that does not divide into its micro-batches (16, 16, 15, 15)
        _vit("vit_s16_ragged_bf16", "bf16", batch=62, micro=4, image=224, patch=16, dim=384, depth=12, heads=6, mlp=1536,
             classes=1000, splits="blocks.6", ranks=2),
        # a decoder with 128-wide heads on sequences of odd length, one sequence to a micro-batch
        _decoder("decoder_wide_heads_bf16", "bf16", batch=4, micro=4, vocab=32000, dim=2048, depth=4, heads=16, ffn=5632,
                 seq=1021, splits="layers.2", ranks=2),
        # one GPU's blocks of ViT-g/14: activations in, an upstream gradient in, head dimension 88
        _share("vit_g14_share_bf16", "bf16", batch=96, micro=4, tokens=257, dim=1408, depth=10, heads=16, mlp=6144),
        # the benchmark's headline: ViT-L/16
        _vit("vit_l16_fp16", "fp16", batch=64, micro=4, image=224, patch=16, dim=1024, depth=24, heads=16, mlp=4096,
             classes=1000, splits="blocks.12", ranks=2),
        # a convolutional stage: ResNet blocks and spatial transformers with cross attention
        _unet("sdxl_stage_fp16", "fp16", batch=4, micro=1, side=32, channels=1280, heads=20, layers=10, context=2048),
        # the largest step: a 1B decoder, 2048-token sequences, four looped stages
        _decoder("llama_1b_bf16", "bf16", batch=16, micro=8, vocab=32000, dim=2048, depth=16, heads=32, ffn=5632, seq=2048,
                 splits="layers.4,layers.8,layers.12", ranks=2),
    ]


def draw(rng):
    while True:
        case = rng.choice((_draw_vit, _draw_decoder, _draw_share, _draw_unet))(rng)
        # a drawn step stays below the largest listed one (fp32 runs at a fraction of the 16-bit rate)
        if work(case)["flops"] <= (2e12 if case["precision"] == "fp32" else 6e13) and _footprint(case) <= 40e9:
            return case


# -- one dict per family ---------------------------------------------------------------------------------------
def _case(name, family, precision, batch, micro, splits, ranks, **sizes):
    case = dict(family=family, precision=precision, batch=batch, micro=micro, splits=splits, ranks=ranks, **sizes)
    if name is not None:
        case["name"] = name
    return case


def _vit(name, precision, *, batch, micro, image, patch, dim, depth, heads, mlp, classes, splits, ranks):
    return _case(name, "vit", precision, batch, micro, splits, ranks, image=image, patch=patch, dim=dim, depth=depth,
                 heads=heads, mlp=mlp, classes=classes)


def _share(name, precision, *, batch, micro, tokens, dim, depth, heads, mlp):
    return _case(name, "share", precision, batch, micro, "", 1, tokens=tokens, dim=dim, depth=depth, heads=heads, mlp=mlp)


def _decoder(name, precision, *, batch, micro, vocab, dim, depth, heads, ffn, seq, splits, ranks):
    return _case(name, "decoder", precision, batch, micro, splits, ranks, vocab=vocab, dim=dim, depth=depth, heads=heads,
                 ffn=ffn, seq=seq)


def _unet(name, precision, *, batch, micro, side, channels, heads, layers, context):
    return _case(name, "unet", precision, batch, micro, "", 1, side=side, channels=channels, heads=heads, layers=layers,
                 context=context)


# -- drawn sizes -----------------------------------------------------------------------------------------------
def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _batches(rng, most):
    """(batch, micro-batches): every other batch leaves a remainder."""
    micro = rng.choice((1, 2, 4, 8))
    per = _log(rng, 1, max(1, most))
    return micro * per + (rng.randrange(micro) if rng.random() < 0.5 else 0), micro


def _boundaries(rng, what, depth):
    """Up to four stages of equal depth, looped over two ranks."""
    stages = rng.choice([s for s in (1, 2, 2, 4) if s <= depth])
    return ",".join("%s.%d" % (what, depth * i // stages) for i in range(1, stages)), min(2, stages)


def _draw_vit(rng):
    precision = rng.choice(("fp32", "fp16", "bf16"))
    heads, hd, depth, patch = _log(rng, 2, 16), rng.choice((32, 64, 64, 80, 88)), rng.randint(1, 8), rng.choice((8, 16))
    batch, micro = _batches(rng, 24)
    splits, ranks = _boundaries(rng, "blocks", depth)
    return _vit(None, precision, batch=batch, micro=micro, image=patch * rng.randint(2, 17), patch=patch, dim=heads * hd,
                depth=depth, heads=heads, mlp=heads * hd * rng.choice((2, 4)), classes=8 * _log(rng, 2, 125), splits=splits,
                ranks=ranks)


def _draw_share(rng):
    heads, hd = _log(rng, 4, 16), rng.choice((64, 64, 80, 88))
    batch, micro = _batches(rng, 24)
    return _share(None, rng.choice(("fp16", "bf16")), batch=batch, micro=micro, tokens=_log(rng, 17, 577), dim=heads * hd,
                  depth=rng.randint(1, 8), heads=heads, mlp=heads * hd * 4)


def _draw_decoder(rng):
    precision = rng.choice(("fp32", "bf16", "bf16", "fp16"))
    heads, hd, depth = _log(rng, 2, 32), rng.choice((64, 64, 96, 128)), rng.randint(1, 8)
    batch, micro = _batches(rng, 4)
    splits, ranks = _boundaries(rng, "layers", depth)
    return _decoder(None, precision, batch=batch, micro=micro, vocab=8 * _log(rng, 64, 4000), dim=heads * hd, depth=depth,
                    heads=heads, ffn=8 * int(heads * hd / 3), seq=_log(rng, 32, 2048), splits=splits, ranks=ranks)


def _draw_unet(rng):
    heads = rng.choice((4, 6, 8, 10, 14, 20))
    batch, micro = _batches(rng, 4)
    return _unet(None, rng.choice(("fp16", "bf16")), batch=batch, micro=micro, side=rng.randint(8, 32), channels=64 * heads,
                 heads=heads, layers=rng.randint(1, 4), context=64 * rng.randint(8, 32))


# -- the program -----------------------------------------------------------------------------------------------
def _model(case):
    fam = case["family"]
    if fam == "vit":
        return vit.VisionTransformer(vit.ViTConfig(image_size=case["image"], patch_size=case["patch"], dim=case["dim"],
                                                   depth=case["depth"], heads=case["heads"], mlp_dim=case["mlp"],
                                                   num_classes=case["classes"]))
    if fam == "share":
        return vit.BlockStack(vit.ViTConfig(dim=case["dim"], depth=case["depth"], heads=case["heads"], mlp_dim=case["mlp"]))
    if fam == "unet":
        c = case["channels"]
        return unet_stage.UNetStage(unet_stage.UNetStageConfig(in_channels=c // 2, channels=c, temb_dim=c,
                                                               context_dim=case["context"], heads=case["heads"],
                                                               layers=case["layers"]))
    return llama.LlamaForCausalLM(llama.LlamaConfig(vocab=case["vocab"], dim=case["dim"], layers=case["depth"],
                                                    heads=case["heads"], ffn=case["ffn"], max_seq=case["seq"]))


def _exec_fn(case, model):
    fam = case["family"]
    if fam == "vit":
        criterion = CrossEntropyLoss(case["classes"])

        def exec_fn(pixels, labels):
            loss = criterion(model(pixels), labels)
            loss.backward()
            return loss.detach()
    elif fam == "share":
        def exec_fn(x, grad_out):
            out = model(x)
            out.backward(grad_out.to(out.dtype))   # the next GPU's blocks send this gradient back
            return out.detach()
    elif fam == "unet":
        def exec_fn(hidden, temb, context, target):
            loss = F.mse_loss(model(hidden, temb, context).float(), target)
            loss.backward()
            return loss.detach()
    else:
        def exec_fn(ids):
            loss = model(ids, ids)                 # next-token cross entropy inside the last stage
            loss.backward()
            return loss.detach()
    return exec_fn


def _batch(case, seed):
    g = torch.Generator("cuda").manual_seed(seed)
    n, fam = case["batch"], case["family"]

    def normal(*shape):
        return torch.randn(*shape, device="cuda", generator=g)

    if fam == "vit":
        return (normal(n, 3, case["image"], case["image"]),
                torch.randint(0, case["classes"], (n,), device="cuda", generator=g))
    if fam == "share":
        shape = (n, case["tokens"], case["dim"])
        return normal(*shape), normal(*shape) * 1e-2
    if fam == "unet":
        c, s = case["channels"], case["side"]
        return normal(n, c // 2, s, s), normal(n, c), normal(n, 77, case["context"]), normal(n, c, s, s)
    return (torch.randint(0, case["vocab"], (n, case["seq"]), device="cuda", generator=g),)


class _Program:
    """The compiled model, its runner and its optimizer.  The parameters and the optimizer's moments of a stage lie in
    one flat tensor each, as in a program that writes checkpoints or averages weights stage by stage."""

    def __init__(self, case):
        torch.manual_seed(1234)
        with torch.device("cuda"):
            model = _model(case)
        self.optimizer = torch.optim.Adam(model.parameters(), lr=LR)
        splits = [s for s in case["splits"].split(",") if s]
        stage, self.stages = 0, [[] for _ in range(len(splits) + 1)]
        for name, p in model.named_parameters():
            while stage < len(splits) and (name + ".").startswith(splits[stage] + "."):
                stage += 1
            self.stages[stage].append(p)
        self.params, self.where = [], []
        for params in self.stages:
            offsets, end = [], 0
            for p in params:
                offsets.append(end)
                end += (p.numel() + 63) // 64 * 64
            flat = torch.zeros(end, device="cuda")
            for p, off in zip(params, offsets):
                flat[off:off + p.numel()].copy_(p.detach().reshape(-1))
                p.data = flat[off:off + p.numel()].view(p.shape)
            self.params.append(flat)
            self.where.append(offsets)
        self.start = [f.clone() for f in self.params]
        self.moments = [[(torch.zeros_like(f), torch.zeros_like(f)) for f in self.params] for _ in range(2)]
        self.active = self.ran_with = 0
        initialize_pfeife()
        option = PipeOption(device_cnt=case["ranks"], batch_cnt=case["micro"], batch_size=-(-case["batch"] // case["micro"]),
                            split_points=splits or None, verbosity="error",
                            mixed_precision=None if case["precision"] == "fp32" else case["precision"])
        self.runner = PartialRunner(option, self.optimizer)
        self.scaler = self.runner.scaler_state_dict()
        self.runner.set_exec_fn(_exec_fn(case, torch.compile(model, backend=partial_compiler)))
        self.restore()
        batch = _batch(case, 99)
        for _ in range(3):      # the first step builds the stage programs, the second captures them
            self.runner.step(*batch)
            self.ran_with = self.active

    def restore(self):
        """Back to the checkpoint every state starts from: first weights, empty moments, first loss scale.  The moments
        go into the pair of tensors that the last step did not use: an optimizer state that is loaded is new tensors."""
        self.optimizer.state_dict()
        self.active = 1 - self.ran_with
        for params, offsets, flat, start, (m, v) in zip(self.stages, self.where, self.params, self.start,
                                                        self.moments[self.active]):
            flat.copy_(start)
            m.zero_()
            v.zero_()
            for p, off in zip(params, offsets):
                view = slice(off, off + p.numel())
                self.optimizer.state[p] = dict(step=torch.tensor(0.0), exp_avg=m[view].view(p.shape),
                                               exp_avg_sq=v[view].view(p.shape))
        self.runner.load_scaler_state_dict(self.scaler)

    def close(self):
        torch.cuda.synchronize()
        self.runner.worker.release()
        self.runner.exec_fn = None
        for p in (p for params in self.stages for p in params):
            p.grad, p.data = None, torch.empty(0)
        self.optimizer.state.clear()
        self.__dict__.clear()
        torch._dynamo.reset()
        gc.collect()
        torch.cuda.empty_cache()


_active = {}    # the one program of this process: {its case: program}


def _program(case):
    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    if key not in _active:
        for old in _active.values():
            old.close()
        _active.clear()
        _active[key] = _Program(case)
    return _active[key]


def prepare(case, seed):
    program = _program(case)
    batch = _batch(case, seed)
    program.restore()
    return program, batch


def run(state):
    program, batch = state
    results = program.runner.step(*batch)
    program.ran_with = program.active
    # Adam's first moments are the weighted sum of the steps' gradients: they hold every parameter's gradient whole
    return {"results": results, "params": program.params, "moments": [m for m, _ in program.moments[program.active]]}


# -- what a step cannot do without -----------------------------------------------------------------------------
def _sizes(case):
    """(parameters, forward operations of one sample)."""
    fam = case["family"]
    if fam in ("vit", "share"):
        d, ff, depth = case["dim"], case["mlp"], case["depth"]
        if fam == "vit":
            grid = (case["image"] // case["patch"]) ** 2
            t, patch = grid + 1, 3 * case["patch"] ** 2
            params = patch * d + d + (t + 1) * d + 2 * d + (d + 1) * case["classes"]
            flops = 2 * grid * patch * d + 2 * d * case["classes"]
        else:
            t, params, flops = case["tokens"], 0, 0
        params += depth * (4 * d * d + 2 * d * ff + 9 * d + ff)
        return params, flops + depth * (8 * t * d * d + 4 * t * d * ff + 4 * t * t * d)
    if fam == "decoder":
        d, ff, depth, t, vocab = case["dim"], case["ffn"], case["depth"], case["seq"], case["vocab"]
        # a causal mask leaves half of the scores
        return 2 * vocab * d + depth * (4 * d * d + 3 * d * ff + 2 * d) + d, \
            t * (depth * (8 * d * d + 6 * d * ff + 2 * t * d) + 2 * d * vocab)
    c, t, ctx, n = case["channels"], case["side"] ** 2, case["context"], case["layers"]
    resnets = [(c // 2, c), (c, c), (c, c), (c, c)]
    params = sum(9 * i * o + 9 * o * o + c * o + 5 * o + 2 * i + (i * o + o if i != o else 0) for i, o in resnets)
    flops = sum(18 * t * i * o + 18 * t * o * o + 2 * c * o + (2 * t * i * o if i != o else 0) for i, o in resnets)
    block = 4 * c * c + 2 * c * c + 2 * ctx * c + 12 * c * c + 17 * c
    per = 2 * t * c * c * 18 + 4 * 77 * ctx * c + 4 * t * t * c + 4 * t * 77 * c
    return params + 3 * (n * block + 2 * c * c + 4 * c), flops + 3 * (n * per + 4 * t * c * c)


def _batch_bytes(case):
    n, fam = case["batch"], case["family"]
    if fam == "vit":
        return n * (12 * case["image"] ** 2 + 8)
    if fam == "share":
        return 3 * 4 * n * case["tokens"] * case["dim"]
    if fam == "unet":
        c, s = case["channels"], case["side"]
        return 4 * n * (c // 2 * s * s + c + 77 * case["context"] + c * s * s)
    return 8 * n * case["seq"]


def _footprint(case):
    """Rough bytes of the activations kept for the backward pass."""
    rows = case["batch"] * {"vit": lambda: (case["image"] // case["patch"]) ** 2 + 1, "share": lambda: case["tokens"],
                            "decoder": lambda: case["seq"], "unet": lambda: case["side"] ** 2}[case["family"]]()
    width = case.get("dim", case.get("channels", 0))
    depth = case.get("depth", 3 * case.get("layers", 0) + 8)
    scores = case["batch"] * case["heads"] * rows / case["batch"] * rows / case["batch"] * 12
    return rows * width * depth * 100 + scores * depth + 8 * rows * case.get("vocab", 0)


def work(case):
    params, forward = _sizes(case)
    # Adam reads and writes parameters and both moments; the batch is read once
    return {"bytes": 24 * params + _batch_bytes(case), "flops": 3 * forward * case["batch"]}


def tolerance(case):
    # 16-bit operands: single results and gradients agree to the rounding of a dozen layers; fp32: to the order of sums
    return {"rel": 1e-4 if case["precision"] == "fp32" else 1e-2}
