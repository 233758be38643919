"""Engine for targets that are served autoregressively in batches (models with ``forward_batch``): prompts are prefilled
together as one packed batch, then the sequences advance in lockstep, one token each, through captured hipGraphs: one per batch
size, and where the best launches depend on how much context there is, a few.  It has the surface the decode loops drive
(``engine``, ``inference``, ``decode_step``, ``clear_kv``) plus ``step`` for batches of named sequences."""
import os

import torch

from .. import ops_tile
from ..models.cache import PagedBatch
from . import graph_infer


class _DecodeBuffers:
    """Static device inputs of the decode step of B sequences.  ``lens`` advances on the device (ops_tile.decode_prep is part of
    the step); the host uploads lengths, page tables and seats when the set of sequences changed, in one asynchronous copy, and sends
    pages that were handed out since as kernel arguments (at 32 sequences some sequence starts a page every other step: three
    copies from pageable memory waited for the device each time, 0.3 ms of it idle)."""

    def __init__(self, cache, B):
        dev = cache.device
        self.B, self.columns = B, cache.columns
        self.ids = torch.zeros(B, dtype=torch.int64, device=dev)
        image = torch.zeros(B * (2 + self.columns), dtype=torch.int32, device=dev)      # lengths | seats | table
        self.lens, self.seat, self.table = self._parts(image)                           # (length or seat -1: idle row)
        self.pos, self.slot, self.klen = (torch.zeros(B, dtype=torch.int32, device=dev) for _ in range(3))
        self.batch = PagedBatch(True, self.pos, self.slot, table=self.table, klen=self.klen, seat=self.seat, max_len=cache.max_budget)
        self.image, self.staged, self.sent = image, torch.zeros(image.shape, dtype=torch.int32, pin_memory=image.is_cuda), None
        self.current, self.known = None, [0] * B                # (births, lengths) the device holds; pages of each row it knows
        self.idle()

    def idle(self):
        """No row is a sequence's: nothing is stored, and everything is sent again afterwards."""
        self.lens.fill_(-1)
        self.seat.fill_(-1)
        self.current = None

    def _parts(self, flat):
        return flat[:self.B], flat[self.B:2 * self.B], flat[2 * self.B:].view(self.B, self.columns)

    def upload(self, cache, seqs):
        """Everything of these sequences; the lengths without the token of this step."""
        if self.sent is not None:
            self.sent.synchronize()                             # (the last copy out of the staging memory is long done)
        lens, seat, table = self._parts(self.staged)
        n, t, s = cache.tables(seqs)
        lens.copy_(n - 1)
        seat.copy_(s)
        table.copy_(t)
        self.image.copy_(self.staged, non_blocking=True)
        if self.image.is_cuda:
            self.sent = torch.cuda.Event()
            self.sent.record()
        self.known = [len(cache.pages[q]) for q in seqs]

    def add_pages(self, cache, seqs):
        """The pages that were handed out to these sequences since the device last heard of them."""
        new = []
        for row, s in enumerate(seqs):
            pages, k = cache.pages[s], self.known[row]
            if len(pages) > k:
                new += [(row, j, pages[j]) for j in range(k, len(pages))]
                self.known[row] = len(pages)
        if new:
            ops_tile.set_pages(self.table, new)


class _DecodeStep:
    """The lockstep decode forward of B sequences: eager, or captured and replayed.  How the launches share the chip may depend on how
    many pages the sequences hold: there is a graph for each of the model's ``decode_form``s (five at most), captured when a step first asks for
    it, as the first one is for a new B."""

    def __init__(self, model, cache, B, use_graph):
        self.model, self.cache, self.buf, self.use_graph = model, cache, _DecodeBuffers(cache, B), use_graph
        self.form = getattr(model, "decode_form", lambda rows, pages, longest: None)                     # (most models have one form)
        self.prepares = getattr(model, "prepares_steps", False)                                          # (decode_prep in the forward's first launch)
        self.graphs = {}                                        # form -> (graph, logits), in one pool: of these only one runs at a time

    def _graph(self, form):
        if form not in self.graphs:                             # warm-up and capture run on idle rows: nothing is stored
            self.buf.idle()
            pool = next(iter(self.graphs.values()))[0].pool() if self.graphs else None
            self.graphs[form] = graph_infer._capture(self._run, (), pool, 2)
        return self.graphs[form]

    def _run(self):
        b = self.buf
        prep = (b.lens, b.table, b.pos, b.slot, b.klen)
        if self.prepares:
            b.batch.prep = prep
        else:
            ops_tile.decode_prep(*prep)
        return self.model.forward_batch(b.ids, b.batch, self.cache)

    def __call__(self, seqs, ids):
        """seqs: the B sequences in order; ids: their next tokens (B,), on the device or the host.  Returns logits (B, V), valid
        until the next call."""
        b, c = self.buf, self.cache
        before = tuple(c.length.get(s, 0) for s in seqs)
        b.batch.pages = sum(n // c.page + 1 for n in before)    # with this step's token
        b.batch.longest = max(before, default=0) // c.page + 1
        graph, logits = self._graph(self.form(b.B, b.batch.pages, b.batch.longest)) if self.use_graph else (None, None)
        c.extend([(s, 1) for s in seqs])
        births = tuple(c.birth[s] for s in seqs)
        if b.current != (births, before):
            b.upload(c, seqs)
        else:
            b.add_pages(c, seqs)
        b.current = (births, tuple(n + 1 for n in before))
        b.ids.copy_(ids)
        if graph is None:
            return self._run()
        graph.replay()
        return logits


class BatchInferenceEngine:
    def __init__(self, model, cache, use_graphs=None):
        self.model, self.kv_cache = model.eval(), cache
        self.use_graphs = os.environ.get("TRIFORCE_DECODE_GRAPH", "1") != "0" if use_graphs is None else bool(use_graphs)
        self._steps = {}

    @property
    def engine(self):                                           # (the decode loops reach model and cache through .engine)
        return self

    def clear_kv(self):
        self.kv_cache.reset()

    # -- named sequences -------------------------------------------------------------------------------------------------
    @torch.inference_mode()
    def step(self, entries, end=()):
        """entries: [(sequence, its next tokens (list of ids), wanted places among them)]; ``end``: sequences that are finished
        after this step.  Returns fp32 logits of the wanted places in order (None when there are none).  A step in which every
        entry brings one token to a sequence that has some is a decode step; all others run the prefill kernels, cut into forwards
        of at most graph_infer.PREFILL_CHUNK tokens."""
        c = self.kv_cache
        names = [s for s, _, _ in entries]
        if len(set(names)) != len(names):
            raise ValueError("a sequence appears twice in one step")
        for s, toks, want in entries:
            if len(toks) == 0:
                raise ValueError(f"sequence {s!r}: no tokens")
            if any(not 0 <= w < len(toks) for w in want):
                raise ValueError(f"sequence {s!r}: a wanted place is outside its tokens")
            if any(not 0 <= t < self.model.vocab_size for t in toks):
                raise ValueError(f"sequence {s!r}: a token id is outside the vocabulary")
        for s in end:
            if s not in c.length and s not in names:
                raise KeyError(f"unknown sequence {s!r}")
        out = None
        if entries:
            if all(len(toks) == 1 and c.length.get(s, 0) > 0 for s, toks, _ in entries):
                logits = self.decode(names, torch.tensor([toks[0] for _, toks, _ in entries], dtype=torch.int64))
                rows = [b for b, (_, _, want) in enumerate(entries) for _ in want]
                if rows:
                    out = logits[rows] if rows != list(range(len(entries))) else logits.clone()
            else:
                out = self._prefill(entries)
        for s in end:
            c.release(s)
        return out

    def _prefill(self, entries):
        c = self.kv_cache
        if c.tokens + sum(len(t) for _, t, _ in entries) > c.max_budget:
            raise IndexError(f"{type(c).__name__} overflow: {c.tokens} + {sum(len(t) for _, t, _ in entries)} > {c.max_budget} tokens")
        at = [0] * len(entries)
        rows = {}                                               # (entry, place) -> logits row
        while True:
            room, portion = graph_infer.PREFILL_CHUNK, []
            for e, (s, toks, want) in enumerate(entries):
                n = min(room, len(toks) - at[e])
                if n > 0:
                    portion.append((e, at[e], n))
                    room -= n
            if not portion:
                break
            ids, plan, keys = [], [], []
            for e, a, n in portion:
                s, toks, want = entries[e]
                places = sorted({w for w in want if a <= w < a + n})
                ids += list(toks[a:a + n])
                plan.append((s, n, [w - a for w in places]))
                keys += [(e, w) for w in places]
                at[e] = a + n
            batch = c.plan_prefill(plan)
            logits = self.model.forward_batch(torch.tensor(ids, dtype=torch.int64).to(c.device), batch, c)
            if keys:
                rows.update({k: logits[j] for j, k in enumerate(keys)})
        out = [rows[(e, w)] for e, (_, _, want) in enumerate(entries) for w in want]
        return torch.stack(out) if out else None

    @torch.inference_mode()
    def decode(self, seqs, ids):
        """One token each for ``seqs``: logits (B, V), valid until the next step of that batch size."""
        B = len(seqs)
        st = self._steps.get(B)
        if st is None:
            st = self._steps[B] = _DecodeStep(self.model, self.kv_cache, B, self.use_graphs)
        return st(seqs, ids.reshape(-1))

    # -- the single-sequence surface of utils/decoding.py ----------------------------------------------------------------
    @torch.inference_mode()
    def inference(self, input_ids, **_):
        """Prompt (or a further portion) of the cache's default sequence -> logits (1, rows, V) like the other engines."""
        return graph_infer.chunked_prefill(lambda ids, last_rows=None: self.model.forward(ids, self.kv_cache, last_rows=last_rows).logits,
                                           input_ids)

    @torch.inference_mode()
    def decode_step(self, input_ids):
        return self.decode([self.kv_cache.DEFAULT], input_ids).unsqueeze(0)
