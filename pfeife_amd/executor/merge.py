"""Stage jobs over several micro-batches.

Micro-batches exist so that the stages of a pipeline can work side by side.  On one GPU that buys nothing: the
same stage over two micro-batches is the same kernels twice, each too short to fill 256 CUs (ViT-L/16, 16
images: 200 tiles of 128x128 for 256 CUs; a looped decoder of 256-wide layers: 64 graph launches of 24 us for
kernels of 3 us).  The samples of a micro-batch do not see each other, so where the buffers of consecutive
micro-batches lie end to end (`BufferPool.stacked`) their launches are ONE launch over all their rows: this
module rewrites the position-aligned launch lists of several micro-batches into one list.

A launch is merged by a rule per kernel (`RULES`) on the call that made it: the operands of the micro-batches
have to follow each other in memory without a gap, everything else has to be the same.  Where that does not
hold (a loss inside the model averages over its micro-batch) the launches stay as they are, one after the
other.  Every row is computed from the same operands as before, products on the tile that suits the longer
operand; gradients that sum over rows (biases, norm weights) add their fp32 terms in another order.

How many micro-batches (`StageWorker.job_rows`): as few as give a job 8192 rows, so that it has up to about twice that many.  Step times on one card in ms, by rows to a
job, sustained: ViT-L/16 (4 x 3152 rows) 36.7 apart, 34.0 in twos, 33.9 all four (31.8 with today's products, in twos and all);
1B decoder (8 x 4096) 205.2 apart, 188.8 in twos, 192.5 in fours; ViT-g share (4 x 6168) 53.7 / 51.7 / 51.9 (today - /
46.0 / 45.0); decoder with wide heads (4 x 1021) 13.1 / - / 10.3; ViT-S fp32 (4 x 788) 9.80 -> 8.64, bf16 with ragged
micro-batches 6.78 -> 5.69; decoder of four looped stages (8 x 256 rows) 3.98 -> 2.95.  Past some 8192 rows the kernels gain
little, and jobs of one rank's forward and another's backward, or user code, no longer run beside each other.
"""
import inspect

import torch


MAX_BATCH = 65535      # products or heads of one launch
MAX_BYTES = 1 << 31    # of one matrix operand


class NoMerge(Exception):
    """The calls do not form one call."""


class Place:
    """Where a micro-batch's part of a stacked buffer lies."""

    __slots__ = ("index", "uniform", "_count", "_size", "_before", "_total")

    def __init__(self, sizes, index, widest, most):
        self.index, self.uniform, self._count = index, len(set(sizes)) <= 1 and widest is None, most
        self._size, self._before = sizes[index], sum(sizes[:index])
        self._total = sum(sizes) if widest is None else widest

    def span(self, numel):
        """(first element, elements in all) for a buffer of `numel` elements here, or (None, None)."""
        if self.uniform:
            return self.index * numel, self._count * numel
        if self._size and numel % self._size == 0:
            per = numel // self._size
            return per * self._before, per * self._total
        return None, None


class MicroBatchLayout:
    """How many samples each micro-batch of a step has, and which consecutive ones share jobs."""

    def __init__(self, sizes, tag):
        self.sizes = list(sizes)
        self.tag = tag               # buffers of slots lowered under the same tag lie end to end
        self.groups = [(i, i + 1) for i in range(len(self.sizes))]
        self.formed = False

    def group(self, mb):
        return next(g for g in self.groups if g[0] <= mb < g[1])

    def form_groups(self, rows_per_sample, target_rows):
        """Consecutive micro-batches share jobs: as few to a job as give it `target_rows` rows."""
        n = len(self.sizes)
        jobs = min(n, max(1, int(sum(self.sizes) * rows_per_sample) // target_rows))
        each = -(-n // jobs)
        self.groups = [(i, min(n, i + each)) for i in range(0, n, each)]
        self.formed = True

    def place(self, mb, in_group=False):
        """in_group: among the micro-batches of its jobs (the jobs' groups use the same memory in turn)."""
        if not in_group:
            return Place(self.sizes, mb, None, len(self.sizes))
        first, end = self.group(mb)
        most = max(b - a for a, b in self.groups)
        if len(set(self.sizes)) <= 1:
            return Place([self.sizes[0]] * most, mb - first, None, most)
        return Place(self.sizes[first:end], mb - first, max(sum(self.sizes[a:b]) for a, b in self.groups), most)


class CallRecorder:
    """A kernel table whose launches remember the call that made them (`launch.call`)."""

    def __init__(self, table):
        self.table = table

    def __getattr__(self, name):
        attr = getattr(self.table, name)
        if name in RULES:
            sig = inspect.signature(attr)

            def prepare(*a, **kw):
                launch = attr(*a, **kw)
                bound = sig.bind(*a, **kw)
                bound.apply_defaults()
                launch.call = (name, bound.arguments)
                return launch
        elif name == "gemm_retiled":
            def prepare(launch, variant):
                new = attr(launch, variant)
                if new is not None:
                    new.call = ("gemm", dict(launch.call[1], variant=variant))
                return new
        elif name == "gemm_group":
            def prepare(launches):
                new = attr(launches)
                new.call = ("gemm_group", dict(launches=list(launches)))
                return new
        else:
            prepare = attr
        self.__dict__[name] = prepare
        return prepare


# -- what the rules are made of ------------------------------------------------------------------------------
def _same(calls, *names):
    for name in names:
        v0 = calls[0][name]
        for c in calls[1:]:
            v = c[name]
            if torch.is_tensor(v0) and torch.is_tensor(v):
                if v.data_ptr() != v0.data_ptr() or v.dtype != v0.dtype:
                    raise NoMerge(name)
            elif type(v) is not type(v0) or v != v0:
                raise NoMerge(name)


def _chain(calls, name, extents):
    """The operand `name` of every call starts where that of the call before ends (`extents`: elements each)."""
    t0 = calls[0][name]
    if t0 is None:
        if any(c[name] is not None for c in calls):
            raise NoMerge(name)
        return None
    at = t0.data_ptr()
    for c, n in zip(calls, extents):
        t = c[name]
        if (t is None or t.dtype != t0.dtype or t.data_ptr() != at
                or t.untyped_storage().data_ptr() != t0.untyped_storage().data_ptr()):
            raise NoMerge(name)
        at += n * t.element_size()
    return t0


def _chains(calls, count, **units):
    """Operands whose extent is `count` (rows, elements, samples) times the given elements."""
    out = {}
    for name, unit in units.items():
        out[name] = _chain(calls, name, [c[count] * (c[unit] if isinstance(unit, str) else unit) for c in calls])
    out[count] = sum(c[count] for c in calls)
    return out


def _heads(calls, name):
    """[B, H, T, hd] operands over all samples."""
    t0 = calls[0][name]
    if t0 is None:
        return _chain(calls, name, [])
    for c in calls:
        if c[name] is None or c[name].shape[1:] != t0.shape[1:] or c[name].stride() != t0.stride():
            raise NoMerge(name)
    _chain(calls, name, [c[name].shape[0] * t0.stride(0) for c in calls])
    return torch.as_strided(t0, (sum(c[name].shape[0] for c in calls),) + tuple(t0.shape[1:]), t0.stride())


def _flat_rule(*operands, same=()):
    def rule(m, calls):
        _same(calls, *same)
        return _chains(calls, "n", **{o: 1 for o in operands})
    return rule


def _gemm(m, calls):
    _same(calls, "a_trans", "b_trans", "N", "lda", "ldb", "ldc", "sa", "sb", "sc", "alpha", "beta", "bias", "round_mid",
          "ld_aux_out", "act", "dact", "ld_aux_in", "ld_res", "unscale_by", "nonfinite_flag")
    c0 = calls[0]
    if "variant" in c0:
        _same(calls, "variant")
    if tuple(c0["batch"]) != (1, 1) or any(tuple(c["batch"]) != (1, 1) for c in calls):
        # one product per head: more samples
        _same(calls, "M", "K")
        if any(c["batch"][1] != c0["batch"][1] or c[o] is not None for c in calls for o in ("aux_out", "aux_in", "residual")):
            raise NoMerge("batch")
        ns = [c["batch"][0] for c in calls]
        if sum(ns) * c0["batch"][1] > MAX_BATCH:
            raise NoMerge("batch")
        return {o: _chain(calls, o, [n * c0[s][0] for n in ns]) for o, s in (("a", "sa"), ("b", "sb"), ("c", "sc"))} | \
            dict(batch=(sum(ns), c0["batch"][1]))
    # (operands are addressed with 32-bit offsets; past 2 GiB of fp32 results the epilogue is the general one)
    if not c0["a_trans"]:
        _same(calls, "K", "b")
        rows = sum(c["M"] for c in calls) + 256
        if max(c0["lda"], 2 * c0["ldc"], 2 * c0["ld_res"], c0["ld_aux_in"], c0["ld_aux_out"]) * 2 * rows >= MAX_BYTES:
            raise NoMerge("size")
        return _chains(calls, "M", a="lda", c="ldc", aux_out="ld_aux_out", aux_in="ld_aux_in", residual="ld_res")
    # a weight gradient that accumulates: a longer reduction; in 16 bits only where each is short (see Merger.lists)
    if c0["a"].dtype != torch.float32 and min(c["K"] for c in calls) >= 64:
        raise NoMerge("weight gradient")
    _same(calls, "M", "c", "aux_out", "aux_in", "residual")
    if not c0["b_trans"] or not c0["beta"] or c0["bias"] is not None or c0["act"] or c0["dact"] or c0["residual"] is not None:
        raise NoMerge("reduction")
    if max(c0["lda"], c0["ldb"]) * 2 * (sum(c["K"] for c in calls) + 256) >= MAX_BYTES:
        raise NoMerge("size")
    return _chains(calls, "K", a="lda", b="ldb")


def _attention(m, calls):
    _same(calls, "scale", "causal")
    kw = {o: _heads(calls, o) for o in calls[0] if o not in ("lse", "delta", "scale", "causal")}
    n = kw["q"].shape[0]
    if n * kw["q"].shape[1] > MAX_BATCH:
        raise NoMerge("batch")
    for o in ("lse", "delta"):
        if o in calls[0]:
            t0 = calls[0][o]
            _chain(calls, o, [c[o].numel() for c in calls])
            kw[o] = torch.as_strided(t0, (n,) + tuple(t0.shape[1:]), t0.stride())
    return kw


def _norm_fwd(m, calls):
    _same(calls, "gamma", "d", "eps", *(["beta"] if "beta" in calls[0] else []))
    return _chains(calls, "rows", x="d", y="d", rstd=1, **({"mean": 1} if "mean" in calls[0] else {}))


def _norm_bwd(m, calls):
    c0 = calls[0]
    fused = "want_wgrad" in c0
    _same(calls, "gamma", "d", *(("want_wgrad", "want_colsum") if fused else ("dgamma", "defer")))
    if "dbeta" in c0:
        _same(calls, "dbeta")
    kw = _chains(calls, "rows", dy="d", x="d", dx="d", dx_add="d", rstd=1, **({"mean": 1} if "mean" in c0 else {}),
                 **({"dx_lp": "d"} if fused else {}))
    if c0["ws"] is not None:
        nb = m.table.norm_bwd_partials(kw["rows"])
        need = nb * (3 if fused and c0["want_colsum"] else 2) * c0["d"]
        kw["ws"] = m.partials(calls, need if fused else max(need, m.table.colreduce_workspace(kw["rows"], c0["d"])), nb)
    return kw


def _colsum(m, calls):
    _same(calls, "cols", "ld", "acc", "defer")
    kw = _chains(calls, "rows", x="ld")
    kw["ws"] = m.partials(calls, m.table.colreduce_workspace(kw["rows"], calls[0]["cols"]),
                          m.table.colsum_partials(kw["rows"]))
    return kw


def _groupnorm(m, calls):
    c0 = calls[0]
    _same(calls, "gamma", "HW", "C", "groups", *(("beta", "eps") if "beta" in c0 else ("dgamma", "dbeta", "defer")))
    per = c0["HW"] * c0["C"]
    kw = _chains(calls, "B", x=per, mean="groups", rstd="groups", **({"y": per} if "y" in c0 else {"dy": per, "dx": per}))
    if "ws" in c0:
        kw["ws"] = m.partials(calls, m.table.groupnorm_workspace(kw["B"], c0["C"], c0["groups"]), kw["B"])
    return kw


def _im2col(m, calls):
    _same(calls, "H", "W", "C", "flip")
    per = calls[0]["H"] * calls[0]["W"] * calls[0]["C"]
    return _chains(calls, "B", src=per, dst=9 * per)


def _softmax(*operands):
    def rule(m, calls):
        _same(calls, "cols", *("ld_" + o for o in operands), *(("scale",) if "scale" in calls[0] else ("q_len", "causal")))
        return _chains(calls, "rows", **{o: "ld_" + o for o in operands})
    return rule


def _glu(*operands):
    def rule(m, calls):
        _same(calls, "act", "cols", *("ld_" + o for o in operands))
        return _chains(calls, "rows", **{o: "ld_" + o for o in operands})
    return rule


def _bias_add(m, calls):
    _same(calls, "bias_len", "rows_per_bias")
    per = calls[0]["rows_per_bias"]
    kw = _chains(calls, "n", x=1, y=1)
    if per:
        if any(c["n"] % (c["bias_len"] * per) for c in calls):
            raise NoMerge("bias")
        kw["bias"] = _chain(calls, "bias", [c["n"] // per for c in calls])
    else:
        _same(calls, "bias")
    return kw


def _copy_strided(m, calls):
    c0 = calls[0]
    _same(calls, "accumulate")
    strides = {o: list(c0[o + "_strides"]) for o in ("src", "dst")}
    if any(list(c[o + "_strides"]) != strides[o] or list(c["sizes"])[1:] != list(c0["sizes"])[1:]
           for c in calls for o in ("src", "dst")):
        raise NoMerge("strides")
    try:                                # the outermost dimension goes on into the next micro-batch
        for o in ("src", "dst"):
            _chain(calls, o, [c["sizes"][0] * strides[o][0] for c in calls])
        if strides["dst"][0] == 0:
            raise NoMerge("dst")
        return dict(sizes=[sum(c["sizes"][0] for c in calls)] + list(c0["sizes"])[1:])
    except NoMerge:
        pass
    if any(list(c["sizes"]) != list(c0["sizes"]) for c in calls) or len(c0["sizes"]) > 5:
        raise NoMerge("sizes")
    step = {}
    for o in ("src", "dst"):            # or the micro-batches are one more dimension
        p = [c[o].data_ptr() for c in calls]
        d = p[1] - p[0]
        if (d < 0 or d % c0[o].element_size() or any(b - a != d for a, b in zip(p, p[1:]))
                or any(c[o].dtype != c0[o].dtype or c[o].untyped_storage().data_ptr() != c0[o].untyped_storage().data_ptr()
                       for c in calls)):
            raise NoMerge(o)
        step[o] = d // c0[o].element_size()
    if step["dst"] == 0:
        raise NoMerge("dst")
    return dict(sizes=[len(calls)] + list(c0["sizes"]), src_strides=[step["src"]] + strides["src"],
                dst_strides=[step["dst"]] + strides["dst"])


def _rope(m, calls):
    _same(calls, "cos_t", "sin_t", "T", "H", "D", "xs", "ys", "inverse", "tab_ld")
    return _chains(calls, "B", x=calls[0]["xs"][0], y=calls[0]["ys"][0])


def _embedding_fwd(m, calls):
    _same(calls, "table", "dim", "vocab")
    return _chains(calls, "n_ids", ids=1, out="dim")


def _embedding_bwd(m, calls):
    _same(calls, "dtable", "dim", "vocab", "padding_idx")
    return _chains(calls, "n_ids", ids=1, dout="dim")


# kernel -> rule(merger, calls) -> the arguments of the one call that differ from the first call's; raises NoMerge
RULES = {
    "gemm": _gemm,
    "attention_fwd": _attention, "attention_bwd": _attention,
    "layernorm_fwd": _norm_fwd, "rmsnorm_fwd": _norm_fwd,
    "layernorm_bwd": _norm_bwd, "rmsnorm_bwd": _norm_bwd, "norm_bwd_fused": _norm_bwd,
    "groupnorm_fwd": _groupnorm, "groupnorm_bwd": _groupnorm,
    "colsum_accumulate": _colsum,
    "softmax_fwd": _softmax("s", "p"), "softmax_bwd": _softmax("dp", "p", "ds"),
    "act_fwd": _flat_rule("x", "y", same=("act",)), "act_bwd": _flat_rule("dy", "x", "dx", same=("act",)),
    "axpby": _flat_rule("a", "b", "out", same=("alpha", "beta")),
    "cast": _flat_rule("src", "dst"), "fill": _flat_rule("dst", same=("value",)),
    "glu_fwd": _glu("gate", "up", "y"), "glu_bwd": _glu("dy", "gate", "up", "dgate", "dup"),
    "bias_add": _bias_add, "copy_strided": _copy_strided, "im2col3x3": _im2col, "rope": _rope,
    "embedding_fwd": _embedding_fwd, "embedding_bwd": _embedding_bwd,
}


class Merger:
    """Merges the launch lists of one stage's programs (one per micro-batch, in micro-batch order)."""

    def __init__(self, table, workspace):
        self.table = table
        self._workspace = workspace    # elements -> fp32 buffer that lives as long as the merged launches
        self._moved = {}               # partial sums that moved: data_ptr -> (buffer, partial rows)

    def partials(self, calls, elements, rows):
        ws = self._workspace(elements)
        for c in calls:
            self._moved[c["ws"].data_ptr()] = (ws, rows)
        return ws

    def _one(self, calls):
        """One launch (or a few) for the calls of a run of micro-batches."""
        name = calls[0].call[0]
        args = [l.call[1] for l in calls]
        if name == "gemm_group":
            rows = list(zip(*(a["launches"] for a in args)))
            if any(len(a["launches"]) != len(rows) for a in args):
                raise NoMerge("members")
            members = [self._one(list(r))[0] for r in rows]
            if len({l.group_key for l in members}) == 1 and all(self.table.gemm_groupable(l) for l in members):
                return [self.table.gemm_group(members)]
            return members
        kw = dict(args[0])
        kw.update(RULES[name](self, args))
        new = getattr(self.table, name)(**kw)
        sums = [getattr(l, "colsum_ws", None) for l in calls]
        if any(s is not None for s in sums):
            cs = self.table.gemm_attach_colsum(new, lambda shape, dtype: self._workspace(shape[0] * shape[1]).view(shape))
            if cs is None or any(s is None for s in sums):
                raise NoMerge("column sums")
            for s in sums:
                self._moved[s.data_ptr()] = (cs[0], cs[2])
        return [new]

    def _try(self, launches):
        moved = dict(self._moved)
        try:
            return self._one(launches)
        except NoMerge:
            self._moved = moved
            return None

    def _position(self, launches):
        """The launches at one place of the lists, merged over runs of micro-batches as long as they go."""
        calls = [getattr(l, "call", None) for l in launches]
        if len(launches) == 1 or any(c is None or c[0] != calls[0][0] for c in calls):
            return list(launches)
        merged = self._try(launches)
        if merged is not None:
            return merged
        moved = dict(self._moved)
        cut = next((i for i in range(1, len(launches)) if self._try(launches[i - 1:i + 1]) is None), None)
        self._moved = moved
        if cut is None:                # (every two would do: too long for one)
            cut = len(launches) // 2
        return self._position(launches[:cut]) + self._position(launches[cut:])

    def lists(self, lists):
        """The merged list, or None.  16-bit weight gradients that accumulate inside the backward jobs (micro-batches of
        different sizes) are not joined: one product over all rows would add its terms in another order than products per
        micro-batch do, and after one update some weights round the other way and every activation follows.
        They need nothing but to run before the job ends: micro-batch by micro-batch there, layers side by side in launches that
        fill the device, they cost as much (ViT-S, 62 images in four micro-batches: 5.63 ms a step, 5.5 joined; where
        they stand, a launch per layer and micro-batch, 7.4)."""
        if len({len(l) for l in lists}) != 1:
            return None
        out, held = [], [[] for _ in lists]
        for pos in zip(*lists):
            parts = [self._weight_gradients(l) for l in pos]
            if len(pos) > 1 and all(parts):
                for h, p in zip(held, parts):
                    h += p
            else:
                out += self._position(list(pos))
        return out + [g for h in held for g in self._grouped(h)]

    def _weight_gradients(self, launch):
        """The products of a launch of 16-bit weight gradients that accumulate, or None."""
        call = getattr(launch, "call", None)
        if call is None or not getattr(launch, "weight_gradients", False) or getattr(self.table, "gemm_retiled", None) is None:
            return None
        members = call[1]["launches"] if call[0] == "gemm_group" else [launch]
        return list(members) if all(self.table.gemm_groupable(l) and l.desc.beta == 1 for l in members) else None

    def _grouped(self, launches):
        """One micro-batch's weight gradients in launches that fill the device on 128x128 tiles (64x64 where all that is
        left is small: BwdCtx._retile_held has both sides' times).  Products into one accumulator (a weight used twice in
        the stage) keep their order: a launch's products run side by side."""
        def tiles(l):
            return ((l.desc.M + 127) // 128) * ((l.desc.N + 127) // 128)

        out, i = [], 0
        while i < len(launches):
            run, n = [launches[i]], tiles(launches[i])
            while i + len(run) < len(launches):
                l = launches[i + len(run)]
                if len(run) == self.table.GEMM_GROUP_MAX or n + tiles(l) > 256 or l.desc.in_dtype != run[0].desc.in_dtype \
                        or any(l.desc.C == r.desc.C for r in run):
                    break
                run.append(l)
                n += tiles(l)
            i += len(run)
            same = [self.table.gemm_retiled(l, 15 if n <= 112 else 8) for l in run]
            if len(run) > 1 and all(l is not None and self.table.gemm_groupable(l) for l in same):
                out.append(self.table.gemm_group(same))
            else:
                out += run
        return out

    def reduces(self, lists):
        """The deferred column reductions [(ws, offset, partial rows, stride, cols, accumulator)] of every
        micro-batch, with partial sums of merged launches in their place."""
        if len({len(l) for l in lists}) != 1:
            return None
        out = []
        for pos in zip(*lists):
            seen = set()
            for ws, off, nb, stride, cols, acc in pos:
                hit = self._moved.get(ws.data_ptr())
                if hit is None:
                    out.append((ws, off, nb, stride, cols, acc))
                elif hit[0].data_ptr() not in seen:
                    seen.add(hit[0].data_ptr())
                    out.append((hit[0], off, hit[1], stride, cols, acc))
        return out
