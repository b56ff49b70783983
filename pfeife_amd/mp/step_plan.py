"""The jobs of a captured step as native job lists, worked out once per capture.

A step alternates between jobs (hipGraph replays on the lanes of the pipeline ranks, with events between them) and user
code (a micro-batch's way to the model; its loss and backward hooks).  Issuing them in one thread adds their host times
up: in a small model's step each is about half, and the GPU waits for both.  Here a native thread issues the jobs
(`Issuer`), and the calling thread waits for it only where user code reads a result:

  * a micro-batch's forward jobs go out as soon as its inputs are in place, while the next micro-batch's user code is
    still on its way to the model, and ahead of the user code of earlier ones: forward jobs read parameters and each
    other only, and with lanes of their own they hold no other job up.  (Without such lanes everything keeps the
    schedule's order.)
  * backward jobs and user code keep the schedule's order among themselves, which fixes the order in which micro-batches
    are summed into a gradient.
  * an event is waited for only if nothing the stream has waited for before implies it, and recorded only if some job
    waits for it.
"""


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
        finals = {i: mb for i, mb in w.last_forward.items()}
        done = {}

        def job(stage, mb, is_fwd):
            prog = w.mbs[mb].stage_programs[stage]
            deps = [done["input", mb]]
            if is_fwd:
                deps += [done[s, mb, True] for s in sorted(sources[stage])]
            else:
                deps += [done[t, mb, False] for t in users_of[stage]] + [done[stage, mb, True]]
                if stage in out_stages:
                    deps.append(done["loss", mb])
            st = lane(stage, is_fwd)
            done[stage, mb, is_fwd] = self._node(st, prog.fwd_graph if is_fwd else prog.bwd_graph, deps)
            if not is_fwd and w.last_backward.get(stage) == mb and w.stack_dw and w.dw_jobs[stage][1] is not None:
                self._node(st, w.dw_jobs[stage][1], [])

        # the step's phases, each a list of nodes: begin, one after each micro-batch's inputs, then job lists and
        # micro-batches ready for user code in turn
        self._begin = [self._node(main, w.begin_graph, [])]
        self._inputs = []
        pending = [(s, mb) for s, mb, f in w.order if f] if early else []
        for bid in range(len(w.mbs)):
            first = len(self._nodes)
            done["input", bid] = self._node(main, None, [])
            while pending and pending[0][1] <= bid:
                job(*pending.pop(0), True)
            self._inputs.append(self._nodes[first:])
        self._turns = []
        first = len(self._nodes)
        for i, (stage, mb, is_fwd) in enumerate(w.order):
            if not (is_fwd and early):
                job(stage, mb, is_fwd)
            if is_fwd and finals.get(i) == mb:
                self._node(main, None, [done[s, mb, True] for s in out_stages])
                self._turns.append((self._nodes[first:], mb))
                first = len(self._nodes)
                done["loss", mb] = self._node(main, None, [])
        self._node(main, None, [n for s, n in self._last.items() if s is not main])
        self._end = self._nodes[first:]

        self._events = []
        for n in self._nodes:
            if n.event:
                n.event = self.issuer.event()
                self._events.append(n.event)
        self._begin, self._end = self._jobs(self._begin), self._jobs(self._end)
        self._inputs = [self._jobs(n) for n in self._inputs]
        self.turns = [(self._jobs(n), mb) for n, mb in self._turns]
        del self._nodes, self._last, self._known, self._turns

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
        self.started = True
        self.issuer.push(self._begin)

    def inputs_ready(self, mb):
        """Micro-batch `mb`'s inputs are on their way on the main stream."""
        self.issuer.push(self._inputs[mb])

    def advance(self, jobs):
        """Issues a turn's jobs: the main stream may then read the outputs of the turn's micro-batch."""
        self.issuer.push(jobs)
        self.issuer.wait()

    def end(self):
        """The rest, and the main stream after every lane."""
        self.advance(self._end)
        self.started = False

    def release(self):
        """After the lanes have been waited for."""
        for ev in self._events:
            self.issuer.destroy_event(ev)
        self._events = []
