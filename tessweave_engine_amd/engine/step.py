"""The step function: one batch of (request, its next tokens) through the model, from the cache.

The reference runs two uniform forwards per scheduler turn, a [B,1] decode
batch and then one [1,T] prompt portion (flow_engine/engine.py:249-260,
model.py:169), and rebuilds and uploads slot lists per layer
(model.py:178, cache.py:98,105-107). Here one call takes any mix of prompt
portions and single decode tokens as ONE flat batch: the metadata of the step
(token ids, positions, cache slots, block tables, lengths, wanted rows) is
packed on the host into a single int32 buffer, uploaded once, and every layer
only reads it. Logits come back in float32 for exactly the rows asked for.

Decode-only steps of a model whose parts are all graph-safe are captured once
per (batch size, length class) into a HIP graph and replayed; only the metadata
upload differs between replays. The length class is the longest sequence of
the step rounded up to a power of two: launch shapes that should follow the
lengths (the number of key ranges of decode attention) follow the class, so an
engine opened for 32,768 tokens that serves 2,000-token requests runs the
launches of a 2,048-token engine.
"""
from __future__ import annotations

from collections import OrderedDict
import ctypes
from dataclasses import dataclass, field
import threading

import numpy as np
import torch

from ..kernels import ops
from ..kernels.lib import library, check
from ..parts.base import GroupStep, StepContext, Workspace


@dataclass
class StepEntry:
    seq: object                      # cache.Sequence
    tokens: list                     # the request's next tokens (at least one)
    want: list = field(default_factory=list)   # indices into tokens whose logits are wanted
    positions: object = None         # None: every position axis counts the request's tokens (computed, computed + 1, ...);
                                     # else one list of len(tokens) position ids per axis of the model's encodings.
                                     # The cache and the causal order go by token order, whatever the ids say.


def _round_up(v, m):
    return (v + m - 1) // m * m


GRAPH_SEGMENT_RUNS = 8       # layer runs per captured graph after the first
MIN_LENGTH_CLASS = 512       # steps whose longest sequence is shorter share one captured graph
SECOND_FORM_MISSES = 16      # a captured step's other form (cut into segments or whole) is captured after so many launches
                             # that wanted it
MAX_GRAPHS = 96              # captured steps kept (one per batch size and length class met); the least recently
                             # replayed one goes first

MAX_VIEWS = 128              # cuts of the metadata buffer kept (see Stepper._cut)


class _Graph:
    """A captured decode step in one or both of two forms, {cut into segments?: (graphs launched one after the other, the
    logits they leave)} (see Stepper._capture).

    BUFFERS names the scratch buffers whose addresses the captures hold, each with its version at the
    time: the captures stay good until one of THOSE is allocated anew (a larger prompt portion growing a
    buffer that only prompt portions use leaves every captured decode step alone)."""

    def __init__(self, generation):
        self.forms, self.generation, self.buffers = {}, generation, {}
        self.missed = 0                      # launches that wanted the form that is not there

    def destroy(self, lib):
        for handles, _ in self.forms.values():
            for handle in handles:
                lib.tw_graph_destroy(handle)


_capturing = threading.local()           # .now: this thread is capturing a step
_let_go_late = []                        # (buffers, readers) of stagings that were collected on a capturing thread


def _wait_for_late():
    while _let_go_late:
        _, readers = _let_go_late.pop()
        for event in readers:
            if event is not None:
                event.synchronize()


class _Staging:
    """Pinned buffers in which steps' metadata waits for the device, taken in turn.

    The kernel that fetches a step's metadata reads its buffer when it runs. The allocator of pinned memory does not know
    of it and would hand the memory to its next taker at once, so the buffers are let go only once their readers are done."""

    def __init__(self, words, device_words, count=4):
        self.buffers = [torch.zeros(words, dtype=torch.int32, pin_memory=True) for _ in range(count)]
        self.arrays = [t.numpy() for t in self.buffers]
        self.uploads = [ops.WordUpload(t, device_words) for t in self.buffers]
        self.readers = [None] * count        # per buffer: an event behind its last reader
        self.next = 0

    def take(self):
        """Index of the next buffer, whose last reader is done."""
        k = self.next
        self.next = (k + 1) % len(self.buffers)
        if self.readers[k] is not None:
            self.readers[k].synchronize()
        return k

    def wait(self):
        for event in self.readers:
            if event is not None:
                event.synchronize()

    def __del__(self):
        try:
            if getattr(_capturing, "now", False):
                _let_go_late.append((self.buffers, self.readers))    # (a wait would end another stepper's capture)
            else:
                self.wait()
        except Exception:       # noqa: BLE001  (half made, or the interpreter is going down)
            pass


class Stepper:
    def __init__(self, model, cache, max_step_tokens=256, max_step_seqs=None, use_graphs=True, max_graphs=MAX_GRAPHS):
        if model.device is None or model.device.type != "cuda":
            raise RuntimeError("the model's weights must be on a GPU: there is no CPU path")
        self.model = model
        self.cache = cache
        self.device = model.device
        self.dtype = model.dtype
        self.workspace = Workspace(self.device)
        self.stream = torch.cuda.Stream(device=self.device)     # captures run here; a step runs on its caller's stream
        self._end, self._end_stream = None, None                 # the end of the last work issued here, and its stream
        self._by_hand = None             # the stream of work that its caller issues by hand (upload, model.forward)
        self.use_graphs = bool(use_graphs) and model.graph_safe_model
        self._defer_sums = bool(getattr(model, "defers_sums", False))
        self.position_axes = max(1, int(getattr(model, "position_axes", 1)))
        self.max_tokens = 0
        self.max_seqs = 0
        self._graphs = OrderedDict()     # (batch size, length class) -> _Graph, least recently replayed first
        self._warm = set()
        self.max_graphs = max(1, int(max_graphs))
        self.token_feed = None
        self.segment_graphs = True
        self._staging = None
        self.steps = 0
        self.graph_replays = 0
        self._reserve(max(1, int(max_step_tokens)), int(max_step_seqs or cache.max_requests))

    # ---- metadata buffers ------------------------------------------------------------
    def _reserve(self, max_tokens, max_seqs):
        """(Re)allocate the metadata buffers for steps of up to MAX_TOKENS rows and MAX_SEQS requests.

        Steps already issued are waited for first (see _Staging)."""
        self._drop_graphs()
        stream = torch.cuda.current_stream(self.device)
        self.synchronize()
        self._follow(stream)
        self.max_tokens, self.max_seqs = max_tokens, max_seqs
        width = self.cache.table_width
        n_groups = len(self.cache.pools)
        sections, offset = {}, 0

        def add(name, count):
            nonlocal offset
            sections[name] = (offset, count)
            offset += _round_up(count, 64)

        add("token_ids", max_tokens)
        add("positions", self.position_axes * max_tokens)
        add("q_start", max_seqs + 1)
        add("kv_len", max_seqs)
        add("state_slots", max_seqs)
        add("state_phase", max_seqs)
        add("kv_page_start", max_seqs + 1)
        add("logit_rows", max_tokens)
        for g in range(n_groups):
            add(f"slots{g}", max_tokens)
            add(f"table{g}", max_seqs * width)
        self._sections, self._meta_ints = sections, offset
        self._meta_dev = torch.zeros(offset, dtype=torch.int32, device=self.device)
        self._staging = None                 # (the old buffers go first)
        self._staging = _Staging(offset, self._meta_dev)
        self._views = OrderedDict()          # (tokens, requests, wanted rows) -> the buffer's sections cut to them, least recently used first
        self._counting = np.arange(max(max_tokens, max_seqs) + 1)
        # a first step on another stream comes behind this stream's work: the clearing of the new buffers, and the model's and
        # the cache's initialisation if they were made here
        self._mark(stream)

    def _dev(self, name, count=None):
        off, cap = self._sections[name]
        return self._meta_dev[off:off + (cap if count is None else count)]

    def _cut(self, n_tokens, n_seqs, n_logits):
        """The metadata buffer's sections as a step of these counts sees them. (They are the same tensors whenever the counts are: a
        decode step's are made once, 25 us of host time.)"""
        key = (n_tokens, n_seqs, n_logits)
        hit = self._views.get(key)
        if hit is None:
            width, axes = self.cache.table_width, self.position_axes
            hit = self._views[key] = (
                self._dev("token_ids", n_tokens), self._dev("positions", axes * n_tokens).view(axes, n_tokens), self._dev("q_start", n_seqs + 1),
                self._dev("kv_len", n_seqs), self._dev("state_slots", n_seqs), self._dev("state_phase", n_seqs),
                self._dev("kv_page_start", n_seqs + 1), self._dev("logit_rows", n_logits),
                [GroupStep(self._dev(f"table{g}", n_seqs * width).view(n_seqs, width), self._dev(f"slots{g}", n_tokens))
                 for g in range(len(self.cache.pools))])
            while len(self._views) > MAX_VIEWS:
                self._views.popitem(last=False)
        else:
            self._views.move_to_end(key)
        return hit

    def _drop_graphs(self):
        if self._graphs:
            torch.cuda.synchronize(self.device)
            lib = library()
            for graph in self._graphs.values():
                graph.destroy(lib)
        self._graphs = OrderedDict()
        self._warm = set()

    def _drop_graph(self, key):
        """Destroy one captured step (it may still be running: wait for the last step first)."""
        graph = self._graphs.pop(key)
        self.synchronize()
        graph.destroy(library())

    def close(self):
        """Let go of captured steps and wait for what has been issued."""
        self._drop_graphs()
        self.synchronize()
        self._staging.wait()

    accepts_token_feed = True

    def set_token_feed(self, feed):
        """FEED (int32, on the device, or None): from now on a token id -1 - k in a step entry stands for
        feed[k] as it is when the step runs, e.g. a token sampled by the step before that the host has not read."""
        if feed is not None and (feed.dtype != torch.int32 or feed.device.type != "cuda" or not feed.is_contiguous()):
            raise ValueError("the token feed must be a contiguous int32 tensor on the model's device")
        same = (feed is None and self.token_feed is None) or \
            (feed is not None and self.token_feed is not None and feed.data_ptr() == self.token_feed.data_ptr()
             and feed.numel() == self.token_feed.numel())
        if not same:
            self._drop_graphs()          # captured steps hold the old pointer
            self.token_feed = feed

    def synchronize(self):
        """Wait for the last step, and for whatever its caller has put on the stepper's own stream or issued by hand."""
        if self._end is not None:
            self._end.synchronize()
        if self._by_hand is not None:
            self._by_hand.synchronize()
        self.stream.synchronize()

    # ---- the step ----------------------------------------------------------------------
    def step(self, entries):
        """Run ENTRIES as one batch; float32 logits [sum(len(e.want)), vocab] in the order of entries and want.

        The returned tensor is scratch memory: read or copy it before the next step.
        """
        entries = list(entries)
        if not entries:
            return torch.empty(0, self.model.vocab_size, dtype=torch.float32, device=self.device)
        ctx, ordered, graphable = self.prepare(entries)
        # The step runs on its caller's stream. On a stream of its own it cost an event and a wait each way, barriers
        # between two hardware queues unless the two streams happened to share one: 18 and 11 us of idle device a step
        # (four layers of the 7B shape at batch 8: 734 us with them).
        stream = torch.cuda.current_stream(self.device)
        self._follow(stream)
        try:
            self._upload(ctx)
            if graphable:
                logits = self._run_graphable(ctx, (ctx.n_seqs, ctx.kv_bound), stream)
            else:
                logits = self.model.forward(ctx)
        finally:
            # one event a step: the staging buffer is free again, and the next step knows what to follow
            self._mark(stream)
            self._staging.readers[ctx.staging_index] = self._end
        self.finish(ordered)
        return logits

    def _mark(self, stream):
        """What has been issued here so far ends where STREAM is now."""
        self._end, self._end_stream = torch.cuda.Event(), stream.cuda_stream
        self._end.record(stream)

    def _follow(self, stream):
        """Work on another stream than the last one's waits for that one's end (they share scratch memory and the metadata
        buffer), and this memory, which may have been allocated for the other stream, is marked as used on this one as well.
        Work issued by hand is waited for up to where its stream is now: its caller went on there behind `upload`."""
        by_hand, self._by_hand = self._by_hand, None
        if self._end is None or self._end_stream == stream.cuda_stream:
            return
        if by_hand is not None:
            stream.wait_stream(by_hand)
        stream.wait_event(self._end)
        for tensor in (self._meta_dev, *self.workspace.buffers.values()):
            tensor.record_stream(stream)

    def finish(self, ordered):
        """Record in the cache that the step's tokens are now held."""
        for e in ordered:
            self.cache.advance(e.seq, e.seq.computed + len(e.tokens))
            e.seq.steps += 1
        self.steps += 1

    def upload(self, ctx):
        """Bring the step's packed metadata to the device (on the current stream): a kernel fetches the parts
        this step filled from the pinned staging buffer, which keeps the step in one queue (a memory copy
        would hand over to the copy engine and back, tens of microseconds of idle queue per step)."""
        stream = torch.cuda.current_stream(self.device)
        self._follow(stream)
        self._upload(ctx)
        self._mark(stream)
        self._by_hand = stream
        self._staging.readers[ctx.staging_index] = self._end

    def _upload(self, ctx):
        k = ctx.staging_index
        if ctx.staging_segments is not None and len(ctx.staging_segments) <= 16:
            self._staging.uploads[k].run(ctx.staging_segments)
        else:
            self._meta_dev.copy_(self._staging.buffers[k], non_blocking=True)

    def prepare(self, entries):
        """Check ENTRIES, take their pages, and build the step's context (host side; nothing runs yet).

        Returns (context, entries in batch order, whether the step can be replayed from a graph).
        """
        vocab, seen = self.model.vocab_size, set()
        feed = self.token_feed.numel() if self.token_feed is not None else 0     # ids -1 .. -feed name fed tokens
        for e in entries:
            if not e.tokens:
                raise ValueError("a step entry needs at least one token")
            if id(e.seq) in seen:
                raise ValueError("a request appears twice in one step")
            seen.add(id(e.seq))
            if e.seq.closed:
                raise ValueError(f"request {e.seq.id!r} is closed")
            if set(map(type, e.tokens)) != {int} or max(e.tokens) >= vocab or min(e.tokens) < -feed:
                raise ValueError(f"request {e.seq.id!r}: token ids must be integers in [0, {vocab})")
            if any(type(w) is not int or w < 0 or w >= len(e.tokens) for w in e.want):
                raise ValueError(f"request {e.seq.id!r}: wanted places must index this step's tokens")
            if e.positions is not None and (len(e.positions) != self.position_axes
                                            or any(len(axis) != len(e.tokens) for axis in e.positions)):
                raise ValueError(f"request {e.seq.id!r}: positions must be {self.position_axes} lists of one id per token")
        n_tokens = sum(len(e.tokens) for e in entries)
        if n_tokens > self.max_tokens or len(entries) > self.max_seqs:
            self._reserve(max(self.max_tokens, _round_up(n_tokens, 256)), max(self.max_seqs, len(entries)))
        for e in entries:
            self.cache.ensure(e.seq, e.seq.computed + len(e.tokens))

        # decode entries (one token) first, then prompt portions; stable
        n_seqs = len(entries)
        n_decode = sum(len(e.tokens) == 1 for e in entries)
        if n_decode == n_seqs:               # (a step that only decodes: everything below counts requests)
            ordered = entries
            q_lens, q_start, seq_of_token = self._counting[1:2].repeat(n_seqs), self._counting[:n_seqs + 1], self._counting[:n_seqs]
            positions = computed = np.array([e.seq.computed for e in ordered], dtype=np.int64)
            kv_len = computed + 1
            token_ids = [e.tokens[0] for e in ordered]
            rows = [i for i, e in enumerate(entries) for _ in e.want]
        else:
            order = sorted(range(n_seqs), key=lambda i: len(entries[i].tokens) != 1)
            ordered = [entries[i] for i in order]
            q_lens = np.array([len(e.tokens) for e in ordered], dtype=np.int64)
            computed = np.array([e.seq.computed for e in ordered], dtype=np.int64)
            q_start = np.zeros(n_seqs + 1, dtype=np.int64)
            np.cumsum(q_lens, out=q_start[1:])
            kv_len = computed + q_lens
            seq_of_token = np.repeat(self._counting[:n_seqs], q_lens)
            positions = self._counting[:n_tokens] - np.repeat(q_start[:-1] - computed, q_lens)
            token_ids = np.concatenate([np.asarray(e.tokens, dtype=np.int64) for e in ordered])
            position_in_order = {orig: pos for pos, orig in enumerate(order)}
            rows = [int(q_start[position_in_order[i]]) + w for i, e in enumerate(entries) for w in e.want]
        state_slots = [e.seq.state_slot for e in ordered]
        n_logits = len(rows)

        # pack the metadata into a pinned buffer and upload it once
        k = self._staging.take()
        host = self._staging.arrays[k]

        segments = []                        # (offset, words) of what this step fills: all that has to travel

        def put(name, values):
            off, _ = self._sections[name]
            host[off:off + len(values)] = values
            segments.append((off, len(values)))

        put("token_ids", token_ids)
        axes = self.position_axes
        if axes == 1 and not any(e.positions is not None for e in ordered):
            put("positions", positions)
        else:
            ids = np.tile(positions, (axes, 1))                  # [axes, n_tokens]; `positions` stays the token order
            for s_index, e in enumerate(ordered):
                if e.positions is not None:
                    ids[:, q_start[s_index]:q_start[s_index + 1]] = np.asarray(e.positions, dtype=np.int64)
            put("positions", ids.reshape(-1))
        put("q_start", q_start)
        put("kv_len", kv_len)
        put("state_slots", state_slots)
        put("state_phase", [e.seq.steps & 1 for e in ordered])
        put("logit_rows", rows)
        page = self.cache.page_size
        kv_page_start = np.zeros(n_seqs + 1, dtype=np.int64)
        np.cumsum((kv_len + page - 1) // page, out=kv_page_start[1:])
        put("kv_page_start", kv_page_start)
        width = self.cache.table_width
        page_of, place = np.divmod(positions, page)
        for g in range(len(self.cache.pools)):
            tables = self.cache.table_rows[g][state_slots]                    # [n_seqs, width]
            pages = tables[seq_of_token, page_of]
            missing = pages < 0
            if missing.any():                # (only behind a window may they be)
                live = positions >= np.repeat(self._first_positions(g, computed), q_lens)
                if missing[live].any():
                    raise RuntimeError("a token's page is not held; the cache manager and the step disagree")
                put(f"slots{g}", np.where(missing, -1, pages * page + place))
            else:
                put(f"slots{g}", pages * page + place)
            off, _ = self._sections[f"table{g}"]
            host[off:off + n_seqs * width] = tables.reshape(-1)
            segments.append((off, n_seqs * width))

        ctx = StepContext()
        ctx.device, ctx.dtype = self.device, self.dtype
        ctx.n_tokens, ctx.n_seqs, ctx.n_decode, ctx.n_logits = n_tokens, n_seqs, n_decode, n_logits
        (ctx.token_ids, ctx.positions, ctx.q_start, ctx.kv_len, ctx.state_slots, ctx.state_phase, ctx.kv_page_start, ctx.logit_rows,
         ctx.groups) = self._cut(n_tokens, n_seqs, n_logits)
        ctx.h_kv_page_start = kv_page_start.tolist()
        ctx.h_q_start = q_start.tolist()
        ctx.h_kv_len = kv_len.tolist()
        ctx.h_state_slots = state_slots
        ctx.max_q_len = int(q_lens[n_decode:].max()) if n_decode < n_seqs else 0
        ctx.max_kv_len = int(kv_len.max())
        ctx.kv_capacity = width * page
        ctx.kv_bound = min(ctx.kv_capacity, max(MIN_LENGTH_CLASS, 1 << max(0, ctx.max_kv_len - 1).bit_length()))
        ctx.max_tokens = self.max_tokens
        ctx.cache, ctx.workspace = self.cache, self.workspace
        ctx.token_feed = self.token_feed
        ctx.defer_sums = self._defer_sums

        graphable = (self.use_graphs and n_decode == n_seqs and n_logits == n_seqs
                     and rows == list(range(n_seqs)))
        ctx.capturing = graphable       # fixed launch shapes in warm-up, capture and replay alike
        ctx.staging_index = k
        ctx.staging_segments = segments
        return ctx, ordered, graphable

    def _first_positions(self, group, computed):
        """Per sequence, the first position whose page a windowed or chunked group must still hold."""
        return self.cache.layout.groups[group].spec.first_position(computed) // self.cache.page_size * self.cache.page_size

    # ---- HIP graphs for decode-only steps ------------------------------------------------
    def _capture(self, ctx, segmented):
        """Capture model.forward(ctx) as a chain of graphs (on the stepper's own stream: nothing runs); returns
        (handles, logits, the scratch buffers whose addresses they hold, each with its version).

        Launching a graph costs host time per node before its first kernel starts. A SEGMENTED step is
        therefore cut after the first layer run and then every GRAPH_SEGMENT_RUNS runs: the first graph
        is short and starts at once, and every later one is launched while its predecessor still runs.
        """
        lib = library()
        stream = self.stream.cuda_stream
        generation = self.workspace.generation
        handles = []
        n_runs = len(self.model.schedule)

        def end_segment():
            handle = ctypes.c_void_p()
            code = lib.tw_graph_end(stream, ctypes.byref(handle))
            if code == 0:
                handles.append(handle)
            return code

        def segment_end(i):
            if segmented and i + 1 < n_runs and (i == 0 or (i + 1) % GRAPH_SEGMENT_RUNS == 0):
                check(end_segment(), "graph capture end")
                check(lib.tw_graph_begin(stream), "graph capture begin")

        _capturing.now = True
        try:
            with torch.cuda.stream(self.stream):
                check(lib.tw_graph_begin(stream), "graph capture begin")
                ctx.segment_end = segment_end
                self.workspace.touched = touched = set()
                try:
                    logits = self.model.forward(ctx)
                except BaseException:
                    end_segment()
                    for handle in handles:
                        lib.tw_graph_destroy(handle)
                    raise
                finally:
                    ctx.segment_end = None
                    self.workspace.touched = None
                check(end_segment(), "graph capture end")
        finally:
            _capturing.now = False
            _wait_for_late()
        if self.workspace.generation != generation:
            for handle in handles:
                lib.tw_graph_destroy(handle)
            raise RuntimeError("a scratch buffer was allocated during graph capture")
        return handles, logits, {key: self.workspace.versions[key] for key in touched}

    def _run_graphable(self, ctx, key, stream):
        """KEY = (batch size, length class) names the captured graph this step can be replayed from."""
        graph = self._graphs.get(key)
        if graph is not None and graph.generation != self.workspace.generation:
            # some scratch buffer was allocated since: only a capture that holds THAT buffer's address is stale
            if self.workspace.holds(graph.buffers):
                graph.generation = self.workspace.generation
            else:
                self._drop_graph(key)
                graph = None
        if graph is None:
            if key not in self._warm:
                # First time at this batch size and length class: run eagerly so every scratch buffer exists.
                self._warm.add(key)
                return self.model.forward(ctx)
            # (the device runs dry while the host captures: the form for an idle one, where cutting is on)
            graph = _Graph(self.workspace.generation)
            self._add_form(graph, ctx, self.segment_graphs)
            self._graphs[key] = graph
            while len(self._graphs) > self.max_graphs:
                self._drop_graph(next(iter(self._graphs)))
        else:
            self._graphs.move_to_end(key)
        # A step that is launched while the step before still runs goes out as one graph: its launch is hidden, and every
        # cut costs about 8 us between two graphs. (The scheduler's lookahead, whose launches always are, turns cutting off.)
        segmented = wanted = self.segment_graphs and (self._end is None or self._end.query())
        if wanted not in graph.forms:
            segmented = not wanted
            graph.missed += 1
        handles, logits = graph.forms[segmented]
        lib = library()
        for handle in handles:
            check(lib.tw_graph_launch(handle, stream.cuda_stream), "graph launch")
        self.graph_replays += 1
        if graph.missed >= SECOND_FORM_MISSES and wanted not in graph.forms:
            self._add_form(graph, ctx, wanted)       # (behind the launch: the device has this step to run meanwhile)
        return logits

    def _add_form(self, graph, ctx, segmented):
        handles, logits, buffers = self._capture(ctx, segmented)
        graph.forms[segmented] = (handles, logits)
        graph.buffers.update(buffers)
