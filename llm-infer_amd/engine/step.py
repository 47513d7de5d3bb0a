"""The description of one step on the device: which tokens run, where they stand in
their sequences, and where their sequences live in the cache."""
from __future__ import annotations

import math

import numpy as np

from ..kernels import ops

PAGE = 64


class StepShared:
    """What the parts of a step share: a value that depends on the step alone (a table of angles, the
    index arrays of a kernel's grid) is made by the first part that asks for it under its key and
    found by the others."""

    def shared(self, key, make):
        store = self.__dict__.setdefault("_shared", {})
        if key not in store:
            store[key] = make()
        return store[key]


class StepContext(StepShared):
    """All index arrays are int32 on the device, uploaded with one copy.

    per token   : token_ids, pos (position in its sequence), tok_slot (its sequence's slot)
    per sequence: seq_slot, seq_qstart (first token of the sequence in this step),
                  seq_qlen (tokens in this step), seq_ctx (context length after the step)
    want_rows   : rows of the step whose logits are asked for
    The host keeps ``host_slots``, ``host_qlens`` and ``host_lens_before`` for parts that plan on the host.
    ``upload=False`` leaves the device arrays out until ``upload()`` is called (a step that is replayed from a
    recording reads them from the recording's own buffer).
    """

    def __init__(self, device, slots, tokens, lens_before, want, upload: bool = True):
        self.n_seqs = len(slots)
        qlens = [len(t) for t in tokens]
        self.n_tokens = sum(qlens)
        self.is_decode = all(q == 1 for q in qlens) and all(l >= 1 for l in lens_before)
        self.max_ctx = max((l + q for l, q in zip(lens_before, qlens)), default=0)
        self.steady_pages = steady_pages([l + q for l, q in zip(lens_before, qlens)])
        self.host_slots, self.host_qlens, self.host_lens_before = list(slots), qlens, list(lens_before)
        qstart = np.concatenate([[0], np.cumsum(qlens)])[:-1] if qlens else np.zeros(0)
        flat = [t for seq in tokens for t in seq]
        pos = [l + j for l, q in zip(lens_before, qlens) for j in range(q)]
        tok_slot = [s for s, q in zip(slots, qlens) for _ in range(q)]
        want_rows = [int(qstart[i]) + w for i, ws in enumerate(want) for w in ws]
        self.n_want = len(want_rows)
        self.device = device
        self.host_tokens, self.host_want_rows = flat, want_rows
        self._fields = [("token_ids", flat), ("pos", pos), ("tok_slot", tok_slot), ("seq_slot", slots),
                        ("seq_qstart", qstart), ("seq_qlen", qlens),
                        ("seq_ctx", [l + q for l, q in zip(lens_before, qlens)]),
                        ("want_rows", want_rows)]
        if upload:
            self.upload()

    def upload(self) -> None:
        """The index arrays onto the device, with one copy."""
        fields, device = self._fields, self.device
        sizes = [len(v) for _, v in fields]
        offs = np.concatenate([[0], np.cumsum([(s + 3) // 4 * 4 for s in sizes])])
        packed = np.zeros(int(offs[-1]) + 4, dtype=np.int32)
        for (_, v), o, s in zip(fields, offs, sizes):
            packed[int(o):int(o) + s] = np.asarray(v, dtype=np.int32)
        dev = ops.upload(packed, device)
        for (name, _), o, s in zip(fields, offs, sizes):
            setattr(self, name, dev[int(o):int(o) + s])
        self._packed = dev

    def decode_splits(self, n_kv_heads: int, n_heads: int) -> int:
        """How many ways the decode attention of a mixer with these heads cuts each sequence's context."""
        return decode_splits(self.n_seqs, n_kv_heads, n_heads, split_bucket(self.max_ctx))

    def page_splits(self, n_kv_heads: int, n_heads: int, head_dim: int = 128, reach: int | None = None) -> int:
        """The same for the kernel whose waves merge inside a workgroup, where a page a split can be worth it (``head_dim``: the
        line between the two depends on it; a mixer that does not say gets that of 128; ``reach``: the most positions that a
        token sees)."""
        return page_splits(self.n_seqs, n_kv_heads, n_heads, split_bucket(self.max_ctx), head_dim, self.steady_pages, reach)

    def steady_splits(self, n_kv_heads: int, n_heads: int, head_dim: int, splits: int, reach: int | None = None) -> bool:
        """Whether so many splits are what ``ops.attention_decode`` calls steady; ``reach``: the most positions that a token sees."""
        return steady_splits(self.n_seqs, n_kv_heads, n_heads, head_dim, splits, self.steady_pages, reach)

    def page_shares(self, n_kv_heads: int, n_heads: int) -> int:
        """The same for the kernels in which a split is a workgroup of four waves."""
        return page_shares(self.n_seqs, n_kv_heads, n_heads, split_bucket(self.max_ctx))


def split_bucket(max_ctx: int) -> int:
    """The most splits that a context of this length is worth (a power of two up to 64): at least two
    pages a split.  It is all that the split count needs to know of the lengths, so a recorded step
    serves every length of one bucket."""
    pages = (max_ctx + PAGE - 1) // PAGE
    s = max(1, min(pages // 2, 64))
    return 1 << (s.bit_length() - 1)


def decode_splits(n_seqs: int, n_kv_heads: int, n_heads: int, bucket: int) -> int:
    """Splits of the context for a decode attention of ``n_seqs`` sequences (a power of two, at most
    ``bucket``), so that the chip is filled."""
    waves = n_seqs * n_kv_heads * ((n_heads // n_kv_heads + 31) // 32)
    # measured on MI355X: 1,024 waves (one a SIMD) fill the chip best; two or four splits are merged inside
    # a workgroup and cost no second kernel
    want = max(1, 1024 // max(1, waves))
    s = max(1, min(want, bucket))
    return 1 << (s.bit_length() - 1)


def steady_pages(lens) -> int:
    """Pages (the nearest power of two) of the contexts of a step whose sequences are all about as long, the shortest at least
    seven eighths of the longest; 0 for other steps, and where that is less than 64.  It is what a recorded step knows beside the
    bucket (``split_bucket``), so it is 0 for fewer than 8 sequences too: their splits are short of a full chip, or of 32 pages up
    to contexts of 64 thousand, and a long conversation is not recorded anew for it."""
    shortest = min(lens, default=0)
    if len(lens) < 8 or shortest == 0 or 8 * shortest < 7 * max(lens):
        return 0
    pages = 1 << round(math.log2((shortest + PAGE - 1) // PAGE))
    return pages if pages >= 64 else 0


def steady_splits(n_seqs: int, n_kv_heads: int, n_heads: int, head_dim: int, splits: int, pages: int, reach: int | None = None) -> bool:
    """Whether a decode step's splits fill the chip with waves that walk long chains of pages to the same end (``pages``:
    ``steady_pages``; ``reach``: the most positions that a token sees), for which ``ops.attention_decode`` has another form of its kernel."""
    # measured on MI355X at 8 and 32 KV heads, all contexts of one length, the other form and this one (figures of heads of 128 beside
    # it, in attention.hip): with 768 waves neither is the faster one (batch 24 at 16,384 264.5 and 278.3, 12 281.6 and 271.1 at
    # 32,768; heads of 64, batch 48 at 8,192 145.7 and 169.1); two splits, which the other form takes as four, from 32 pages each
    # on (64 at 4,096 194.6 and 191.3, of 64 96.4 and 93.4), one from 64 on (128 at 2,048 197.3 and 198.8, at 4,096 365.3 and
    # 361.2), more from as many bytes on as 32 pages of heads of 128 (of 64, 16 at 16,384 96.7 and 98.8, at 32,768 187.9 and
    # 184.4).  Other heads: the other form (64 at 8,192, of 96 271 and 272, of 80 254 and 258; of 32 by a third, of 256 three times)
    if head_dim not in (64, 112, 128) or splits != decode_splits(n_seqs, n_kv_heads, n_heads, 64):
        return False
    if reach:
        pages = min(pages, reach // PAGE)
    waves = splits * n_seqs * n_kv_heads * ((n_heads // n_kv_heads + 31) // 32)
    return waves >= 1024 and pages >= splits * {1: 64, 2: 32}.get(splits, 4096 // head_dim)


def page_splits(n_seqs: int, n_kv_heads: int, n_heads: int, bucket: int, head_dim: int, pages: int = 0, reach: int | None = None) -> int:
    """Splits for the softmax decoder's decode kernel (``ops.attention_decode``): as ``decode_splits``, but down to one page a
    split (a bucket stands for 2 to 4 times as many pages, the first for 1 to 3), at most 64.  Heads of up to 160 are not split
    beyond four, which merge inside a workgroup, for more waves than half the chip's SIMDs, and those below 128 not into eight.
    ``pages``, ``reach``: as for ``steady_splits``."""
    # measured on MI355X with tiles of 32 rows, us with half as many splits and with these.  Heads of 128, 8 KV heads, batch 1 at 40
    # tokens 6.2 and 6.1, at 100 7.5 and 6.3, at 250 7.6 and 6.7, at 500 8.2 and 8.6, at 777 10.3 and 9.2 (with a soft cap and gates 12.5
    # and 10.3), at 1,000 9.9 and 9.0, at 2,000 11.3 and 10.4, at 4,000 14.1 and 11.7; batch 32 at 250 10.7 and 10.5.  Not taken
    # (what more would take): 128, batch 16 at 500 11.3 (13.1), at 900 15.5 (17.9), batch 4 at 4,000 18.1 (18.6), batch 8 at 1,900
    # 17.0 (17.8), batch 2 at 8,000 18.6 (19.6); 64, batch 1 at 500 7.6 (8.6), at 900 8.5 (8.7), batch 8 at 500 8.6 (10.2), at 900
    # 11.0 (10.6); 96, batch 1 at 700 8.1 (9.0), batch 8 at 900 12.1 (11.8); 160, 4 KV heads, 64 splits at 8,000 19.0 (20.0).  Heads
    # of 256, 2 KV heads, whose pages are longer: batch 1 at 500 30 and 18, batch 32 at 1,000 67 and 49
    # Two splits where four would make more than 1,024 waves: four after all, since two waves of the tile of 16 rows share a SIMD,
    # unless the two are steady.  8 KV heads, us in two and four: heads of 128, batch 40 at 16 to 528 tokens 18.2 and 18.2, 48 18.7 and
    # 18.7, 64 20.8 and 20.9, 64 at 900 57.0 and 55.7, at 1,056 65.1 and 61.8, at 1,000 to 8,192 245.7 and 238.9; heads of 64,
    # 48 at 16 to 528 11.1 and 10.9, 64 at 1,056 33.3 and 30.0.  More than 512 waves in one split keep the one (open: us in one,
    # two and four of heads of 128, 65 at 16 to 528 23.0, 21.4 and 20.8, 96 26.3, 25.5 and 27.7, 128 38.8, 38.6 and 38.7; 96 at 1,000
    # 72.7, 76.7 and 78.9, 128 at 2,048 183.1, 186.5 and 191.0; 32 KV heads, 17 at 2,000 107.5, 109.5 and 112.0)
    few, many = (decode_splits(n_seqs, n_kv_heads, n_heads, min(b, 64)) for b in (bucket, 2 * bucket))
    waves = many * n_seqs * n_kv_heads * ((n_heads // n_kv_heads + 31) // 32)
    if few == many == 2 and head_dim <= 128 and head_dim % 32 == 0 and n_heads <= 16 * n_kv_heads:
        return 2 if steady_splits(n_seqs, n_kv_heads, n_heads, head_dim, 2, pages, reach) else 4
    return few if head_dim <= 160 and many > 4 and (waves > 512 or (few == 4 and head_dim < 128) or (many == 64 and head_dim > 128)) else many


def page_shares(n_seqs: int, n_kv_heads: int, n_heads: int, bucket: int) -> int:
    """Shares of a token's keys for the decode kernels of differential and latent attention, whose share is a workgroup of four
    waves that merge inside it (a power of two): down to one page each as ``page_splits``, one for the shortest contexts,
    and no more workgroups than CUs."""
    # measured on MI355X, us.  One share: latents of 256 / 192 (16 heads, batch 8) at 64 keys 9.6 (10.7 in two, with the kernel that
    # merges them), at 128 10.2 (11.4), at 192 12.2 (11.3); two maps of 64 with values of 128 (32 / 8 heads, batch 4) at 64 9.9
    # (12.9), at 128 10.6 (13.6), at 192 13.9 (12.7).  Longer contexts, shares that make 256 workgroups (and twice as many): latents
    # of 32 heads, batch 32 at 2,000 24.7 (34.3), batch 64 at 1,000 24.8 (33.9), batch 16 at 4,000 23.9 (33.7); two maps, batch 4
    # at 2,000 19.6 (23.9), batch 8 at 600 18.7 (22.1), batch 16 at 600 22.9 (26.4), batch 32 at 300 19.6 (27.2).  Fewer than
    # that, a page a share (and two): latents batch 1 at 300 13.2 (14.7), at 600 13.3 (15.0), at 4,000 14.6 (15.6), but
    # at 2,000, two pages after all, 14.5 (13.6)
    groups = n_seqs * n_kv_heads * ((n_heads // n_kv_heads + 31) // 32)
    s = 1 if bucket == 1 else max(1, min(2 * bucket, 64, 256 // max(1, groups)))
    return 1 << (s.bit_length() - 1)
