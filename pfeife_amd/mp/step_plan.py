"""The jobs of a captured step as native job lists, worked out once per capture.

A step begins when every micro-batch's user code has reached the model: until then user code may change weights, read or
drop gradients, and nothing of the step has touched them.  From there it alternates between jobs (hipGraph replays on the
lanes of the pipeline ranks, with events between them) and user code (a micro-batch's loss and backward hooks).  Issuing
them in one thread adds their host times up, and the GPU waits for both.  Here a native thread issues the jobs
(`Issuer`), and the calling thread waits for it only where user code reads a result:

  * with lanes of their own, forward jobs are issued up to the end of the next micro-batch while this one's user code
    runs: they read parameters and each other only, and hold no other job up.  (Without such lanes everything keeps the
    schedule's order.)
  * backward jobs and user code keep the schedule's order among themselves, which fixes the order in which micro-batches
    are summed into a gradient.
  * an event is waited for only if nothing the stream has waited for before implies it, and recorded only if some job
    waits for it.

Against the same graphs issued job by job in the calling thread: two-layer ViT on four 32x32 images, two micro-batches
1.14 -> 0.88 ms; decoder of four looped stages, eight micro-batches of 256 tokens 5.3 -> 3.85 ms; ViT-S on 62 images in
bf16 6.76 -> 6.69 ms, on 16 in fp32 9.83 -> 9.77 ms.

Where all micro-batches of a stage are one job, what follows on each other anyway is one graph (`_whole`): the decoder 2.74 -> 2.43 ms, the
two-layer ViT 1.15 -> 1.08.
"""

# Operations of a step's weight-gradient jobs up to which all its backward jobs are one graph.  us apart / as one: decoder of 256 columns, 1.4e10
# operations 2430 / 2190, six-layer ViT of 384 in fp32, 6e9, 1856 / 1810; ViT-S on 16 images, 1.3e11, bf16 2625 / 2652, fp32 7754 / 7952; decoder of
# 1024 columns, 2.4e11, 2589 / 2621
SMALL_DW = 3e10


class _Node:
    __slots__ = ("stream", "idx", "graph", "waits", "event", "known")

    def __init__(self, stream, idx, graph):
        self.stream, self.idx, self.graph = stream, idx, graph
        self.waits = []      # nodes of other streams
        self.event = None    # True: some node waits for this one; then the event
        self.known = {}      # stream -> last node of it that is complete when this one starts


class StepPlan:
    def __init__(self, worker):
        self.worker = worker
        self.issuer = worker.issuer
        self.started = False
        self._graphs = []    # captured here
        self._nodes = []
        self._last = {}      # stream -> its last node
        self._known = {}     # stream -> {other stream: index of its last node known to be complete}
        w, pg = worker, worker.part_graph
        main = w.stream_obj
        early = w.lanes is not None and w.lane_mode == "rankdir"
        lane = (lambda s, f: w.lanes[w._lane_key(s, f)]) if w.lanes is not None else (lambda s, f: main)
        sources = {s.idx: {src[0] for src in s.input_source if src is not None} for s in pg.nodes.values()}
        users_of = {s: sorted(t for t in sources if s in sources[t]) for s in sources}
        out_stages = sorted({ref[0] for ref in pg.outputs if isinstance(ref[0], int)})
        done = {}
        everything = [(s, m, f) for s in pg.nodes for m in w.mbs for f in (True, False)]
        forward, backward = self._whole(everything)
        # (after the inputs' copies, on the same stream)
        begin = self._node(main, forward if forward is not None else w.begin_graph, [])
        if forward is not None:
            done.update({k: begin for k in everything if k[2]})

        def job(stage, mb, is_fwd):
            j = w.jobs[stage, mb]
            if mb != (j.first if is_fwd else j.last) or (stage, mb, is_fwd) in done:
                return           # part of the job that runs at another place
            if not is_fwd and backward is not None:
                node = self._node(main, backward, [begin])    # (and after every micro-batch's loss, on the same stream)
                done.update({k: node for k in everything if not k[2]})
                return
            deps = [begin]
            for m in j.mbs:
                if is_fwd:
                    deps += [done[s, m, True] for s in sorted(sources[stage])]
                else:
                    deps += [done[t, m, False] for t in users_of[stage]] + [done[stage, m, True]]
                    if stage in out_stages:
                        deps.append(done["loss", m])
            st = lane(stage, is_fwd)
            node = self._node(st, j.prog.fwd_graph if is_fwd else j.prog.bwd_graph, deps)
            done.update({(stage, m, is_fwd): node for m in j.mbs})
            if not is_fwd and w.last_backward.get(stage) == mb and w.stack_dw and w.dw_jobs[stage][1] is not None:
                self._node(st, w.dw_jobs[stage][1], [])

        # the step's phases, each a list of nodes: begin, then job lists and micro-batches ready for user code in turn
        finals = [i for i in range(len(w.order)) if i in w.last_forward]     # of each micro-batch in turn
        ahead = [(i, s, mb) for i, (s, mb, f) in enumerate(w.order) if f] if early else []

        def take():
            nonlocal first
            nodes, first = self._nodes[first:], len(self._nodes)
            return nodes

        def forward_through(i):
            while ahead and ahead[0][0] <= i:
                job(*ahead.pop(0)[1:], True)

        first, turns = 0, []
        self._begin = take()
        for i, (stage, mb, is_fwd) in enumerate(w.order):
            if not (is_fwd and early):
                job(stage, mb, is_fwd)
            if is_fwd and w.last_forward.get(i) == mb:
                forward_through(i)
                self._node(main, None, [done[s, mb, True] for s in out_stages])
                needed = take()
                later = finals[len(turns) + 1:]
                if later:
                    forward_through(later[0])
                turns.append((needed, take(), mb))
                done["loss", mb] = self._node(main, None, [])
        self._node(main, None, [n for s, n in self._last.items() if s is not main])
        self._end = take()

        self._events = []
        for n in self._nodes:
            if n.event:
                n.event = self.issuer.event()
                self._events.append(n.event)
        self._begin, self._end = self._jobs(self._begin), self._jobs(self._end)
        self.turns = [((self._jobs(n), self._jobs(a)), mb) for n, a, mb in turns]
        del self._nodes, self._last, self._known

    def _whole(self, everything):
        """-> (graph of the step's begin and all forward jobs, graph of all backward and weight-gradient jobs), None where they stay apart.
        With all micro-batches in one job per stage the forward jobs are a chain: one graph in place of as many launches, events and
        waits (each some 25 us of the host, and a gap on the GPU).  So are the backward jobs, but for the weight gradients, which run
        beside the next stage's: apart where those are worth more than the launches."""
        w = self.worker
        if any(len(j.mbs) < len(w.mbs) for j in w.jobs.values()):
            return None, None
        progs = [w.jobs[s, min(w.mbs)].prog for s in sorted(w.part_graph.nodes)]
        forward = w.begin_launches() + [l for p in progs for l in p.fwd]
        forward = self._capture(forward)
        dw = {s: w.dw_jobs[s][0] if w.stack_dw else [] for s in w.part_graph.nodes}
        backward = None
        if sum(getattr(l, "flops", None) or 0.0 for ls in dw.values() for l in ls) <= SMALL_DW:
            backward = self._capture([l for s in sorted(dw, reverse=True) for l in list(w.jobs[s, min(w.mbs)].prog.bwd) + list(dw[s])])
        return forward, backward

    def _capture(self, launches):
        self._graphs.append(self.worker.kernels.capture(launches, self.worker.stream()))
        return self._graphs[-1]

    def _node(self, stream, graph, deps):
        known = self._known.setdefault(stream, {})
        prev = self._last.get(stream)
        n = _Node(stream, prev.idx + 1 if prev is not None else 0, graph)
        # (what the latest node of a stream implies needs no wait: look at those first)
        for d in sorted(set(deps), key=lambda d: -sum(d.known.values()) - d.idx):
            if d.stream is stream or known.get(d.stream, -1) >= d.idx:
                continue
            n.waits.append(d)
            d.event = True
            for s, i in list(d.known.items()) + [(d.stream, d.idx)]:
                known[s] = max(known.get(s, -1), i)
        n.known = dict(known)
        self._last[stream] = n
        self._nodes.append(n)
        return n

    def _jobs(self, nodes):
        return self.issuer.jobs([(n.graph, n.stream.cuda_stream, [d.event for d in n.waits], n.event or None)
                                 for n in nodes if n.graph is not None or n.waits or n.event])

    # -- one step ---------------------------------------------------------------------
    def begin(self):
        """The inputs of all micro-batches are on their way on the main stream."""
        self.started = True
        self.issuer.push(self._begin)

    def advance(self, turn):
        """Issues a turn's jobs: the main stream may then read the outputs of the turn's micro-batch."""
        needed, ahead = turn
        ticket = self.issuer.push(needed)
        self.issuer.push(ahead)
        self.issuer.wait(ticket)

    def end(self):
        """Hands over the rest, and the main stream after every lane; -> what returns once all of it has been issued."""
        self.issuer.push(self._end)
        return self._settle

    def _settle(self):
        self.issuer.wait()
        self.started = False

    def release(self):
        """After the lanes have been waited for."""
        for ev in self._events:
            self.issuer.destroy_event(ev)
        self._events = []
        for graph in self._graphs:
            self.worker.kernels.destroy_graph(graph)
        self._graphs = []
