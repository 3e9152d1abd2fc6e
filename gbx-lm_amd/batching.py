"""Ragged step batches and the slot scheduler of models that hold per-sequence state in slots (models/cache.py:SequenceSlots).

A step is a list of (sequence, its next tokens): sequences that start and sequences that go on by one token mix freely, each
with its own position.  The tokens of a step are laid out back to back -- no padding rows exist, so nothing a sequence computes
depends on the lengths of its neighbours -- and every kernel finds a token's sequence, slot and position through the small
descriptor tables built here once per step (one host-to-device copy).

``BatchScheduler`` is the engine above it: it owns the caches, hands slots out and takes them back, runs a step through
``model.forward_tokens`` and the output head on the rows that are asked for, and generates for several prompts at once
(``generate``) with the same sampler interface as ``generate_step``.
"""
from __future__ import annotations

from array import array
from dataclasses import dataclass, field
from operator import index
from typing import Callable, Dict, Iterable, List, Optional, Sequence, Tuple

import torch

from . import env, graphs


# Rows up to which the host writes a step's tables entry by entry: the device's kernel starts behind a copy of its own (us a table, host's time / until it is there, host |
# device: 1 row 17 / 20 | 22 / 35, 64 rows 24 / 27 | 23 / 34, 200 38 / 42 | 23 / 35, 8 192 1 009 / 1 023 | 23 / 35; 32 sequences of one row 39 / 42 | 30 / 42).
HOST_ROWS = 64


@dataclass
class StepBatch:
    """One step's layout.  Host lists (one item per sequence of the step) and their device images."""
    slot: List[int]
    pos0: List[int]                 # position of the sequence's first new token
    n_new: List[int]
    total: int                      # tokens of the step
    seq: torch.Tensor               # int32 [B, 4]: slot, pos0, n_new, first row of the sequence in the step
    tok: torch.Tensor               # int32 [T, 2]: sequence of the step a row belongs to, its position
    q_tile: int = 0                 # query rows per tile of ``tiles``
    tiles: Optional[torch.Tensor] = None   # int32 [n_tiles, 2]: sequence of the step, first row of the tile inside it
    keys_of: Dict[int, Tuple[int, int]] = field(default_factory=dict, repr=False, compare=False)       # ``tile_keys``: the same for every layer of the step

    @property
    def decode_only(self) -> bool:
        return all(n == 1 for n in self.n_new)

    def tile_keys(self, window: int) -> Tuple[int, int]:
        """Keys that a tile's rows see together under ``window``: the most of any tile, and their sum over the tiles."""
        if window not in self.keys_of:
            q = self.q_tile
            keys = [min(p + min(t + q, n), window + min(q, n - t) - 1) for p, n in zip(self.pos0, self.n_new) for t in range(0, n, q)] if q else [0]
            self.keys_of[window] = max(keys), sum(keys)
        return self.keys_of[window]

    @staticmethod
    def build(slot: Sequence[int], pos0: Sequence[int], n_new: Sequence[int], device, q_tile: int = 128) -> "StepBatch":
        if q_tile < 1:
            raise ValueError("a query tile holds at least one row")
        rows, seq, tile0, n_tiles = 0, [], [], 0
        for s, p, n in zip(slot, pos0, map(index, n_new)):
            if n <= 0:
                raise ValueError("a sequence of a step brings at least one token")
            if p + n > 1 << 31:
                raise RuntimeError("a position does not fit the tables' 32 bits")
            seq += (s, p, n, rows)
            tile0.append(n_tiles)
            rows += n
            n_tiles += -(-n // q_tile)
        nb, dev = len(tile0), torch.device(device)
        if dev.type == "cuda" and rows > HOST_ROWS:
            from . import _lib, ops
            head = torch.tensor(seq + tile0, dtype=torch.int32).pin_memory().to(dev, non_blocking=True)
            tables = torch.empty((2 * (rows + n_tiles),), dtype=torch.int32, device=dev)
            tok, tiles = tables[:2 * rows].view(rows, 2), tables[2 * rows:].view(n_tiles, 2)
            _lib.check_mixers(_lib.mixers().gbxm_step_tables(head.data_ptr(), head.data_ptr() + 16 * nb, tok.data_ptr(), tiles.data_ptr(), nb, rows, n_tiles, q_tile,
                                                             ops._stream_ptr(tables.device)))
            return StepBatch(list(slot), list(pos0), list(n_new), rows, head[:4 * nb].view(nb, 4), tok, q_tile, tiles)
        tok = [v for b, (p, n) in enumerate(zip(pos0, n_new)) for i in range(n) for v in (b, p + i)]
        tiles = [v for b, n in enumerate(n_new) for t in range(0, n, q_tile) for v in (b, t)]
        packed = torch.tensor(seq + tok + tiles, dtype=torch.int32)
        if dev.type == "cuda":
            packed = packed.pin_memory().to(dev, non_blocking=True)
        return StepBatch(list(slot), list(pos0), list(n_new), rows, packed[:4 * nb].view(nb, 4), packed[4 * nb:4 * nb + 2 * rows].view(rows, 2), q_tile,
                         packed[4 * nb + 2 * rows:].view(n_tiles, 2))


class _DecodeGraph:
    """One decode step (every sequence brings one token) of a fixed set of slots, captured in a HIP graph.  Tokens and the step's
    descriptor tables live in one static device buffer that a single host-to-device copy refreshes before each replay; the
    launches, their grids and every pointer they read are the same from step to step, only positions and tokens change."""

    def __init__(self, sched: "BatchScheduler", slots: Tuple[int, ...]):
        self.slots = slots
        b = len(slots)
        dev = sched.device
        # int64 words: tokens [b] | seq [b, 4] as int32 pairs | tok [b, 2] | tiles [b, 2]
        self.words = b + 2 * b + b + b
        self.static = torch.zeros((self.words,), dtype=torch.int64, device=dev)
        self.pinned = [torch.zeros((self.words,), dtype=torch.int64, pin_memory=True) for _ in range(2)]
        self.views = []                                  # per host buffer: tokens, and the places of the positions; the rest never changes
        for host in self.pinned:
            a64 = host.numpy()
            a32 = a64.view("int32")
            seq, tok, tiles = a32[2 * b:6 * b].reshape(b, 4), a32[6 * b:8 * b].reshape(b, 2), a32[8 * b:10 * b].reshape(b, 2)
            seq[:, 0], seq[:, 2], seq[:, 3] = slots, 1, range(b)
            tok[:, 0] = tiles[:, 0] = range(b)
            self.views.append((a64[:b], seq[:, 1], tok[:, 1]))
        self.copied = [torch.cuda.Event() for _ in range(2)]           # (an event that was never recorded has passed)
        self.turn = 0
        i32 = self.static.view(torch.int32)
        self.tokens = self.static[:b]
        self.batch = StepBatch(list(slots), [0] * b, [1] * b, b, i32[2 * b:6 * b].view(b, 4), i32[6 * b:8 * b].view(b, 2), 128,
                               i32[8 * b:10 * b].view(b, 2))
        self.graph = None
        self.logits = None                               # rows of the output head (``BatchScheduler._head``) ...
        self.whole = False                               # ... as it was when they were captured: whether ``_finish`` has to follow
        self.at: Optional[List[int]] = None              # positions that the static tables hold

    def fill(self, tokens: Sequence[int], pos0: Sequence[int]) -> None:
        k = self.turn % 2
        self.turn += 1
        self.copied[k].synchronize()                     # the copy that last read this host buffer has run
        words, seq_pos, tok_pos = self.views[k]
        try:
            words[:] = array("q", tokens)                # (as in an eager step: device tensors by their value)
        except TypeError:                                # not whole numbers: torch's conversion
            words[:] = torch.tensor(tokens, dtype=torch.long).numpy()
        seq_pos[:] = tok_pos[:] = pos0
        self.static.copy_(self.pinned[k], non_blocking=True)
        self.copied[k].record(torch.cuda.current_stream(self.static.device))
        self.batch.pos0 = self.at = list(pos0)

    def advance(self, tokens: torch.Tensor, rows: int) -> None:
        """The next token of every sequence, from the device: one small launch instead of a copy from the host that has read them there first.  What is no row of an
        embedding of ``rows`` goes on as token 0."""
        from . import _lib, ops
        b = len(self.slots)
        _lib.check_mixers(_lib.mixers().gbxm_step_advance(tokens.data_ptr(), tokens.element_size(), rows, self.static.data_ptr(), self.batch.seq.data_ptr(),
                                                          self.batch.tok.data_ptr(), b, ops._stream_ptr(self.static.device)))
        self.batch.pos0 = self.at = [p + 1 for p in self.at]

    def run(self, sched: "BatchScheduler") -> torch.Tensor:
        if self.graph is None:
            torch.cuda.synchronize(sched.device)
            g = torch.cuda.CUDAGraph()
            self.whole = sched._whole_head()
            with graphs.capture(g):
                self.logits = sched._head(sched.model.forward_tokens(self.tokens, self.batch, sched.caches), self.whole)
            self.graph = g
        self.graph.replay()
        return self.logits


class BatchScheduler:
    """Sequences in slots, stepped together.  ``step`` takes what each live sequence brings next and returns the logits of the rows
    that are asked for; ``release`` gives a finished sequence's slot back.  ``max_tokens`` bounds the tokens live sequences may hold
    (a request past it is refused before anything is written)."""

    def __init__(self, model, max_tokens: Optional[int] = None):
        self.model = model
        self.caches = model.make_cache()
        self.slots = self.caches[0].slots
        self.slots.length[0] = -1                       # make_cache hands out slot 0 for the one-sequence loop; nothing holds it here
        self.max_tokens = max_tokens
        self.slot_of: Dict[object, int] = {}
        self.device = next(model.parameters()).device
        # decode-only steps of a set of slots that keeps coming back are replayed from a HIP graph (captured at its third step)
        self.use_graphs = self.device.type == "cuda" and env.flag("GBX_STEP_GRAPH")
        self._graphs: Dict[Tuple[int, ...], _DecodeGraph] = {}
        self._seen: Dict[Tuple[int, ...], int] = {}
        self._buffers = None

    def _whole_head(self) -> bool:
        """Whether a model's logits are ``finish_logits`` of ``head_rows``, which then may be finished where they are read."""
        from .models.step_model import RaggedStepModel as R
        m, t = self.model, type(self.model)
        return (isinstance(m, R) and t.logits is R.logits and t.finish_logits is R.finish_logits and not {"logits", "finish_logits"} & vars(m).keys())

    def _head(self, hidden: torch.Tensor, whole: bool) -> torch.Tensor:
        return self.model.head_rows(hidden) if whole else self.model.logits(hidden)

    def _finish(self, rows: torch.Tensor, whole: bool) -> torch.Tensor:
        """The logits of ``_head``'s rows, by what was decided when these were made (a wrapper put over ``logits`` since then has not seen them)."""
        from .models.step_model import RaggedStepModel
        return RaggedStepModel.finish_logits(self.model, rows) if whole else rows

    def position(self, seq_id) -> int:
        return self.slots.length[self.slot_of[seq_id]]

    def release(self, seq_id) -> None:
        self.slots.release(self.slot_of.pop(seq_id))

    @torch.no_grad()
    def step(self, entries: Sequence[Tuple[object, Sequence[int]]], want: Optional[Sequence[Sequence[int]]] = None) -> torch.Tensor:
        """``entries``: (sequence id, next tokens); an id not seen before starts a sequence at position 0.  ``want[i]``: places among
        entry i's tokens whose logits are returned (default: the last one), in the order of entries and places.  Returns fp32
        [wanted, vocab]."""
        return self._step(entries, want)

    def _step(self, entries, want=None, raw: bool = False):
        """``raw``: the output head's rows as they are, of every entry's last token, and whether they are still to be finished; the caller is done with them before the
        next step, whose replay may overwrite them."""
        if not entries:
            return torch.empty((0, 0))
        new_tokens = sum(len(t) for _, t in entries)
        if self.max_tokens is not None and self.slots.live_tokens() + new_tokens > self.max_tokens:
            raise RuntimeError(f"step would hold {self.slots.live_tokens() + new_tokens} tokens, more than max_tokens={self.max_tokens}")
        if len({i for i, _ in entries}) != len(entries):
            raise ValueError("a sequence appears twice in one step")
        for seq_id, _ in entries:
            if seq_id not in self.slot_of:
                self.slot_of[seq_id] = self.slots.acquire()
        slot = [self.slot_of[i] for i, _ in entries]
        pos0 = [self.slots.length[s] for s in slot]
        n_new = [len(t) for _, t in entries]
        if self.use_graphs and all(n == 1 for n in n_new) and len(slot) <= 256:
            g = self._graph_step(tuple(slot), [ts[0] for _, ts in entries], pos0)
            if g is not None:
                for s in slot:
                    self.slots.length[s] += 1
                if raw:
                    return g.logits, g.whole
                buffer, logits = g.logits, self._finish(g.logits, g.whole)
                rows = [i for i in range(len(slot)) if want is None or len(want[i])]
                if any(p != 0 for i in rows if want is not None for p in want[i]):
                    raise ValueError("a wanted place lies outside the entry's tokens")
                if not rows:
                    return torch.empty((0, self.model.args.vocab), dtype=torch.float32, device=self.device)
                if len(rows) == len(slot):
                    return logits.float() if logits.dtype != torch.float32 else logits.clone() if logits is buffer else logits      # (the graph's buffer is overwritten by the next replay)
                return logits.index_select(0, torch.tensor(rows, dtype=torch.long, device=self.device)).float()
        batch = StepBatch.build(slot, pos0, n_new, self.device)
        try:
            flat = array("q")
            for _, ts in entries:
                flat.extend(ts)
            tokens = torch.frombuffer(flat, dtype=torch.long)
        except TypeError:                               # not whole numbers: torch's conversion
            tokens = torch.tensor([t for _, ts in entries for t in ts], dtype=torch.long)
        if self.device.type == "cuda":
            tokens = tokens.pin_memory().to(self.device, non_blocking=True)
        hidden = self.model.forward_tokens(tokens, batch, self.caches)
        for s, n in zip(slot, n_new):
            self.slots.length[s] += n
        rows, first = [], 0
        for i, n in enumerate(n_new):
            places = [n - 1] if want is None else want[i]
            for p in places:
                if not 0 <= p < n:
                    raise ValueError("a wanted place lies outside the entry's tokens")
                rows.append(first + p)
            first += n
        if not rows:
            return torch.empty((0, self.model.args.vocab), dtype=torch.float32, device=self.device)
        idx = torch.tensor(rows, dtype=torch.long, device=self.device)
        whole = self._whole_head()
        out = self._head(hidden.index_select(0, idx), whole)
        return (out, whole) if raw else self._finish(out, whole).float()

    def _current_graph(self, slots: Tuple[int, ...], longest: int) -> Optional["_DecodeGraph"]:
        """The captured step of these slots, dropped with all others where a table it reads has moved."""
        for c in self.caches:                            # tables without a window grow on the host, never inside a replay
            if hasattr(c, "ensure"):
                c.ensure(longest)
        buffers = tuple(b.data_ptr() if b is not None else 0 for c in self.caches
                        for b in (c.buffers() if hasattr(c, "buffers") else (c.keys,)))
        if buffers != self._buffers:                     # rings were (re)allocated: every captured pointer is stale
            self._graphs.clear()
            self._seen.clear()
            self._buffers = buffers
        return self._graphs.get(slots)

    def _step_ahead(self, ids: Sequence[object], tokens: torch.Tensor):
        """The next step of the sequences ``ids``, enqueued before the host has seen their tokens: (the tokens on their way to the host, the event behind that copy,
        the output head's rows, whether they are still to be finished), or None where that step has to be laid out on the host."""
        if not (self.use_graphs and 0 < len(ids) <= 256 and isinstance(tokens, torch.Tensor) and tokens.device == self.device and tokens.dtype in (torch.int64, torch.int32)
                and tokens.numel() == len(ids) and all(i in self.slot_of for i in ids)):
            return None
        if self.max_tokens is not None and self.slots.live_tokens() + len(ids) > self.max_tokens:
            return None
        table = getattr(self.model, "token_rows", None)              # (tokens that nobody has looked at yet stay inside the embedding)
        if table is None:
            return None
        slots = tuple(self.slot_of[i] for i in ids)
        at = [self.slots.length[s] - 1 for s in slots]
        # tables grow, and captured steps are dropped, behind the host's look at the tokens: a sequence that ends here needs no row more, and nothing runs then
        longest = max(at) + 2
        if not all(c.holds(longest) if hasattr(c, "holds") else not hasattr(c, "ensure") for c in self.caches):
            return None
        g = self._current_graph(slots, longest)
        if g is None or g.graph is None or g.at != at:
            return None
        tokens = tokens.contiguous()
        host = torch.empty((len(ids),), dtype=tokens.dtype, pin_memory=True)
        host.copy_(tokens, non_blocking=True)
        there = torch.cuda.Event()
        there.record(torch.cuda.current_stream(self.device))
        g.advance(tokens, table)
        rows = g.run(self)
        for s in slots:
            self.slots.length[s] += 1
        return host, there, rows, g.whole

    def _graph_step(self, slots: Tuple[int, ...], tokens: Sequence[int], pos0: Sequence[int]) -> Optional["_DecodeGraph"]:
        """Replay (or, at the third step of this set of slots, capture) the decode graph; None: run the step eagerly."""
        g = self._current_graph(slots, max(pos0) + 1)
        if 0 in self._buffers:
            return None
        if g is None:
            self._seen[slots] = self._seen.get(slots, 0) + 1
            if self._seen[slots] < 3:
                return None
            if len(self._graphs) >= 8:                   # a few live compositions at most: drop the oldest
                self._graphs.pop(next(iter(self._graphs)))
            g = self._graphs[slots] = _DecodeGraph(self, slots)
            self._seen.pop(slots, None)
        g.fill(tokens, pos0)
        g.run(self)
        return g

    @torch.no_grad()
    def generate(self, prompts: Sequence[Sequence[int]], max_tokens: int = 64,
                 sampler: Optional[Callable[[torch.Tensor], torch.Tensor]] = None,
                 stop_tokens: Iterable[int] = ()) -> List[List[int]]:
        """Generate for several prompts at once: one ragged prompt step, then one token per live sequence and step.  A sequence that
        samples a stop token (or reaches ``max_tokens``) leaves the batch and frees its slot; the others go on.  ``sampler`` maps
        log-probabilities [n, vocab] to token ids [n] (default: greedy), as in ``generate_step``."""
        from .mixer_ops import log_probabilities
        sampler = sampler or (lambda lp: torch.argmax(lp, dim=-1))
        stop = set(stop_tokens)
        ids = [object() for _ in prompts]
        out: List[List[int]] = [[] for _ in prompts]
        live = list(range(len(prompts)))
        feed = {i: list(prompts[i]) for i in live}
        rows, whole = None, False                       # the output head's rows of a step that is under way already, and whether they are still to be finished
        # A step that someone put in the place of the scheduler's is called as it is, from the first on that is not under way.
        plain = lambda: getattr(self.step, "__func__", None) is _PLAIN_STEP
        while live:
            # log-probabilities are a tensor of their own: the plain step's rows need not outlive its next replay
            if rows is None and plain():
                rows, whole = self._step([(ids[i], feed[i]) for i in live], raw=True)
            if rows is not None:
                logprobs = log_probabilities(rows, self.model.logit_scale if whole and self.model.logit_scale is not None else 1.0)
            else:
                logprobs = log_probabilities(self.step([(ids[i], feed[i]) for i in live]))
            toks = sampler(logprobs).reshape(-1)
            # Where every sequence goes on, unless a token ends it, the next step is enqueued behind the tokens before the host reads them: the chip does not wait for the host's
            # turn (some 40 us a step).  A sequence that a token has ended then has run one step too many, in a slot that is given back.
            ahead = self._step_ahead([ids[i] for i in live], toks) if plain() and all(len(out[i]) + 1 < max_tokens for i in live) else None
            if ahead is None:
                values, rows = toks.tolist(), None
            else:
                host, there, rows, whole = ahead
                there.synchronize()
                values = host.tolist()
            nxt, kept = [], []
            for at, (i, t) in enumerate(zip(live, values)):
                out[i].append(int(t))
                if int(t) in stop or len(out[i]) >= max_tokens:
                    self.release(ids[i])
                elif ahead is not None and not 0 <= t < self.model.token_rows:
                    raise ValueError(f"the sampler chose token {t}, which is neither a stop token nor one of the model's {self.model.token_rows}")
                else:
                    feed[i] = [int(t)]
                    nxt.append(i)
                    kept.append(at)
            if rows is not None and len(kept) < len(live) and kept:
                rows = rows.index_select(0, torch.tensor(kept, dtype=torch.long, device=rows.device))
            live = nxt
        return out


_PLAIN_STEP = BatchScheduler.step
