"""Short prompts as recorded steps.

A step of a few tokens on a model of many layers is bound by the host: some three hundred kernel
launches take longer to enqueue than the device needs to run them.  Such a step (at most
``MAX_TOKENS`` tokens in at most ``MAX_SEQS`` sequences) is therefore recorded into a HIP graph, keyed by
the numbers of rows it runs, and replayed.  The rows are the step's tokens, sequences and wanted places, each
rounded up to a bucket (``decode.batch_bucket``); what a step does not fill is padding that changes no
result: padded tokens sit on the cache's scratch slot (they write the null page and belong to no sequence,
so no attention tile covers them), padded sequences have no tokens, padded wanted places repeat row 0 and
are cut off the result.  Everything a recorded step reads of the step lies in one device buffer of index
arrays that is refilled with one copy before each replay; page tables and lengths are updated outside the
graph, as for decoding.  The reference replays a recorded graph per token in the same spirit
(src/model/model.cu:11-22).

Only parts that say so are recorded (``prefill_recordable``): a part that plans on the host from the step's
lengths (``ctx.host_qlens``) would have its plan frozen into the graph.

A step of one token for each sequence, called for by itself instead of through a decode runner, is recorded
likewise on models of up to ``MAX_STEP_BYTES``, of this library's own parts, that the runner records (a decode
step of theirs plans nothing on the host).  It is not padded: a recording is for so many sequences and wanted
rows and the bucket of context lengths, and runs the kernels that the eager step runs, so that a call gives the
same bits the first time and the tenth.  An eager one takes the host 0.7 to 0.95 ms on models of four layers, the
device 0.35 to 0.6.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from ..kernels import ops
from .decode import _GraphContext, batch_bucket, recording
from .step import StepShared, split_bucket

MAX_TOKENS = 512          # a longer step keeps the device busy longer than the host needs to enqueue it
MAX_SEQS = 16
# largest model (bytes of its matrices) whose steps of one token are recorded: beyond, the step is the device's (the 8B shape, batch
# 1: 3.2 ms eagerly, the host's 3.0 of them meanwhile, 3.15 replayed), and a recording of many layers takes 10 ms
MAX_STEP_BYTES = 6 << 30
# what an engine keeps of each kind, prompts and steps of one token; the least recently used goes first.  Kept apart: a loop of steps
# over many batch sizes and context lengths would push every prompt's recording out, each time with a wait for the device
MAX_RECORDED = 32


class _RecordedContext(StepShared):
    """The step description of a recorded prefill step: slices of the one device buffer."""
    is_decode = False

    def __init__(self, fields, n_tokens, n_seqs, n_want, device):
        self.n_tokens, self.n_seqs, self.n_want, self.device = n_tokens, n_seqs, n_want, device
        for name, t in fields.items():
            setattr(self, name, t)


def _matrix_bytes(model) -> int:
    return sum(math.prod(p.shape) for p in model.params().values() if len(p.shape) == 2) * model.dtype.itemsize


def _only_own_parts(model) -> bool:
    """True if every part of the model is this library's: a part from outside may read of a step what a recorded one does not
    have (``host_slots``), and so far only a decode runner recorded it."""
    stack = list(model.children())
    while stack:
        part = stack.pop()
        if type(part).__module__.split(".")[0] != __name__.split(".")[0]:
            return False
        stack += list(part.children()) if hasattr(part, "children") else []
    return True


class PrefillRecorder:
    """The recorded prefill steps of one engine (which is handed in with every call: the engine holds this
    object, and a reference back would keep both alive until the garbage collector finds the cycle)."""

    def __init__(self):
        self.graphs = {}                   # prompts: key -> "seen" | (graph, logits, index arrays on the device)
        self.step_graphs = {}              # steps of one token: key -> (graph, logits, index arrays)
        self._step_seen = {}               # those called for once or twice: key -> "once" | "seen"
        self.counts = {"eager": 0, "recorded": 0, "replayed": 0}
        self._stream = None                # where the last recording was replayed

    # -- which steps ---------------------------------------------------------------
    def takes(self, eng, ctx) -> bool:
        """A step of whole prompts (or chunks of them) that is small enough, on a model whose parts can all
        be recorded."""
        if ctx.n_want == 0 or ctx.n_tokens > MAX_TOKENS or ctx.n_seqs > MAX_SEQS:
            return False
        if ctx.is_decode:
            if getattr(self, "_steps_ok", None) is None:
                self._steps_ok = (_matrix_bytes(eng.model) <= MAX_STEP_BYTES and eng.model.recordable()
                                  and _only_own_parts(eng.model))
            return self._steps_ok
        if getattr(self, "_model_ok", None) is None:
            model = eng.model
            mixers = [m for ms in model.layer_mixers for m in ms]
            self._model_ok = model.recordable() and all(getattr(m, "prefill_recordable", False) for m in mixers)
        return self._model_ok

    # -- the buffer of index arrays ------------------------------------------------
    @staticmethod
    def _layout(rows, seqs, wants):
        tiles = -(-rows // ops.Q_TILE) + seqs            # at most this many attention tiles
        sizes = [("token_ids", rows), ("pos", rows), ("tok_slot", rows), ("seq_slot", seqs), ("seq_qstart", seqs),
                 ("seq_qlen", seqs), ("seq_ctx", seqs), ("want_rows", wants), ("tile_seq", tiles), ("tile_q0", tiles)]
        layout, at = {}, 0
        for name, n in sizes:
            layout[name] = (at, n)
            at += (n + 3) // 4 * 4
        return layout, at

    @staticmethod
    def _fill(ctx, layout, total, scratch):
        """The step's index arrays with their padding, as one int32 array."""
        packed = np.zeros(total, dtype=np.int32)

        def put(name, values, pad):
            at, n = layout[name]
            packed[at:at + n] = pad
            packed[at:at + len(values)] = values
        qlens, before = ctx.host_qlens, ctx.host_lens_before
        qstart = np.concatenate([[0], np.cumsum(qlens)])[:-1]
        put("token_ids", ctx.host_tokens, 0)
        put("pos", [b + j for b, q in zip(before, qlens) for j in range(q)], 0)
        put("tok_slot", [s for s, q in zip(ctx.host_slots, qlens) for _ in range(q)], scratch)
        put("seq_slot", ctx.host_slots, scratch)
        put("seq_qstart", qstart, 0)
        put("seq_qlen", qlens, 0)
        put("seq_ctx", [b + q for b, q in zip(before, qlens)], 0)
        put("want_rows", ctx.host_want_rows, 0)
        tile_seq, tile_q0 = ops.prefill_tiles(qlens)
        put("tile_seq", tile_seq, 0)
        put("tile_q0", tile_q0, 1 << 30)                  # a tile that begins beyond its sequence does nothing
        return packed

    @staticmethod
    def _fill_decode(ctx):
        """The same for a step of one token a sequence: tokens, positions, contexts, slots and wanted rows, each array on a
        multiple of four elements (16 bytes)."""
        n = (ctx.n_seqs + 3) // 4 * 4
        packed = np.zeros(4 * n + ctx.n_want, dtype=np.int32)
        before = np.array(ctx.host_lens_before)
        for i, values in enumerate((ctx.host_tokens, before, before + 1, ctx.host_slots, ctx.host_want_rows)):
            packed[i * n:i * n + len(values)] = values
        return packed

    @staticmethod
    def _decode_context(buf, rows, wants, bucket, pages=0):
        n = (rows + 3) // 4 * 4
        fields = {name: buf[i * n:] for i, name in enumerate(("tokens", "pos", "ctx", "slots", "rows"))}
        ctx = _GraphContext(fields, rows, bucket, pages)
        ctx.n_want, ctx.want_rows = wants, fields["rows"][:wants]
        return ctx

    # -- the step --------------------------------------------------------------------
    def run(self, eng, ctx):
        """The logits of the step [n_want, vocab], or None if this step is to be run eagerly (the first time
        its key is seen, or the second)."""
        rows, seqs, wants, bucket = ctx.n_tokens, ctx.n_seqs, ctx.n_want, None
        if ctx.is_decode:
            bucket = (split_bucket(ctx.max_ctx), ctx.steady_pages)
        else:
            rows, seqs = batch_bucket(rows, MAX_TOKENS), batch_bucket(seqs, MAX_SEQS)
            wants = batch_bucket(wants, rows)
        key = (rows, seqs, wants, bucket)
        graphs = self.step_graphs if ctx.is_decode else self.graphs
        entry = graphs.pop(key, None) or self._step_seen.pop(key, None)
        # a recording takes some milliseconds: a step of one token is recorded when it comes for the third time (one behind a prompt
        # and one at a request's end are no loop)
        if entry is None or entry == "once":
            if ctx.is_decode:
                self._step_seen[key] = "seen" if entry else "once"
            else:
                graphs[key] = "seen"
            self.counts["eager"] += 1
            self._trim()
            return None
        if ctx.is_decode:
            packed = self._fill_decode(ctx)
        else:
            layout, total = self._layout(rows, seqs, wants)
            packed = self._fill(ctx, layout, total, eng.cache.scratch_slot)
        # a recording's index arrays and results are its own: a step on another stream waits for the one before it
        stream = torch.cuda.current_stream(eng.device)
        if self._stream is not None and stream != self._stream:
            stream.wait_stream(self._stream)
        self._stream = stream
        if entry == "seen":
            buf = torch.from_numpy(packed).to(eng.device)
            graph = torch.cuda.CUDAGraph()
            with recording(graph):
                if ctx.is_decode:
                    rec = self._decode_context(buf, rows, wants, *bucket)
                else:
                    fields = {name: buf[at:at + n] for name, (at, n) in layout.items()}
                    tiles = {"tile_seq": fields.pop("tile_seq"), "tile_q0": fields.pop("tile_q0"), "n_tiles": layout["tile_seq"][1]}
                    rec = _RecordedContext(fields, rows, seqs, wants, eng.device)
                    rec.shared(ops.PREFILL_TILES_KEY, lambda: tiles)
                logits = eng.model.forward(rec, eng.cache)
            entry = (graph, logits, buf)
            self.counts["recorded"] += 1
        else:
            entry[2].copy_(torch.from_numpy(packed))
            self.counts["replayed"] += 1
        entry[0].replay()
        graphs[key] = entry
        self._trim()
        return entry[1][:ctx.n_want].clone()

    def _trim(self):
        for graphs in (self.graphs, self.step_graphs):
            while len(graphs) > MAX_RECORDED:
                old = next(iter(graphs))
                if graphs[old] != "seen":
                    torch.cuda.synchronize()             # it may still be running
                del graphs[old]
        while len(self._step_seen) > 16 * MAX_RECORDED:
            del self._step_seen[next(iter(self._step_seen))]
