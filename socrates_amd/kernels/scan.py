"""Wrapper of the kernels in ``csrc/scan.hip``: the recurrences with a matrix state per head over long portions, 64
tokens at a time on the matrix cores, and the rule that says when. The library is compiled and loaded when a model
first asks for it."""

from __future__ import annotations

from ctypes import c_int, c_longlong, c_void_p

import torch

from .build import load_library
from .common import _SCAN_SIGNATURES, _check, _declare, _ptr

CHUNK = 64
HEAD, STEP, CHANNEL, BONUS = range(4)          # what the decays are: see csrc/scan.hip
NO_LIMIT = (1 << 31) - 1                       # the walks' sequences: those of fewer tokens than this


def _tiles(D, Dv):
    """Elements of a head's state in tiles of 16 channels by 16 columns, an even number of them along the columns."""
    return -(-D // 16) * 16 * -(-Dv // 32) * 32


class Scan:
    # Tokens of a step's longest portion from which it may be taken in chunks (0: never). Measured in us, walk -> chunks, at
    # the heads of a 4B-sized layer: 64 tokens: retention 30 -> 41, gated linear attention 33 -> 54, wkv 30 -> 41,
    # ssd 33 -> 31; 100 tokens: 43 -> 41, 47 -> 54, 33 -> 41, 48 -> 33; 300: 142 -> 50, 158 -> 63, 80 -> 41, 127 -> 48.
    # The gated delta rule, whose chunk costs more and whose walk is faster: 200 tokens 59 -> 69, 256: 73 -> 71, 300: 83 -> 72.
    scan_from, delta_scan_from = 160, 256
    scan_scratch = 1 << 30           # bytes of scratch that one launch over all chunks may take; beyond, in rounds

    def _scan_lib(self):
        lib = getattr(self, "_scan_library", None)
        if lib is None:
            lib = self._scan_library = load_library("scan")
            _declare(lib, _SCAN_SIGNATURES)
        return lib

    def _in_chunks(self, ctx, D, least=None):
        """Whether a step's longest portion is one for chunks: of some length, and with keys of ``D`` whose queries, keys
        and decays of a chunk fit LDS. ``least``: tokens, in place of ``scan_from``."""
        return 0 < (self.scan_from if least is None else least) <= ctx.max_q_len and D <= 128

    def _chunks_from(self, ctx, D, cols, work=1.0, least=None, token=None, serial=0.0, busy=7e-4, start=32.0, chunk=0.0145):
        """Tokens from which on a sequence of the step is taken in chunks (0: all walk): of all such lines, the one whose estimate
        is least. A chunk costs the same however few of its tokens there are, so decoding rows walk beside a portion in
        chunks. With ``cols`` blocks of 16 columns in the states of all heads, in us:
        a walk: 12 and the most of ``token`` for every token of its longest sequence, ``serial`` for those and ``busy`` for every
        token and block, its states' bytes; chunks: ``start`` and ``chunk`` for every chunk and block; 15 for the launch of a walk
        beside them. Fitted to 20 heads of 128 x 128, 10 of 128 x 256, 40 of 64 x 64 and 80 of 128 x 64; measured, all walk -> all
        in chunks -> walks beside chunks: 160 tokens beside 50 decoding rows: retention 93 -> 154 -> 83; 500 beside 60: wkv
        158 -> 187 -> 89, linear attention 270 -> 263 -> 114; 2,000 beside 60: retention 890 -> 299 -> 156, ssd 1,149 -> 606 -> 286.

        A step of few tokens is bound by the host's launches, of which chunks have two more per layer and a walk beside them
        another, so there the kernels' gain is none of the step's: the mean of the longest sequence and of all tokens
        in chunks has to reach ``work`` times ``scan_from``, beside a walk 5 / 4 of that. Whole steps, us, walk -> chunks
        throughout (-> beside a walk): wkv and ssd (9 / 5), 6 layers: 256 tokens 1,977 -> 1,989, 300 2,115 -> 2,014, 2 x 162 1,951
        -> 2,022, 2 x 200 2,103 -> 2,042, 260 to 78 in five 2,854 -> 2,610, 300 beside 30 decoding rows 2,940 -> 3,002 -> 3,040,
        500 beside 7 2,887 -> 2,383 -> 2,442; linear attention (23 / 20), 8 layers: 162 2,214 -> 2,375, 200 2,480 -> 2,348, 2 x 162 2,622 -> 2,423, 250
        beside 7 2,926 -> 2,709 -> 2,816; retention (1), 6 layers: 162 2,894 -> 2,819, 162 beside 60 3,864 -> 3,999 -> 3,925, 250 beside 60
        4,410 -> 4,533 -> 4,323.
        A step that does not say its lengths on the host is taken in chunks whole."""
        if not self._in_chunks(ctx, D, least):
            return 0
        enough = 2 * work * (self.scan_from if least is None else least)
        step = self._lengths_and_lines(ctx)
        if step is None:
            return int(2 * ctx.max_q_len >= enough)
        lens, lines = step
        key = (D, cols, work, token, serial, busy, start, chunk)
        if key not in lines:
            token = 0.12 + 0.0028 * D if token is None else token

            def walk(longest, tokens, n):
                return 12.0 + max(token * longest, serial * longest + busy * cols * tokens, cols * D * 128 / 4.8e6 * n)
            left, chunks, n = sum(lens), 0, len(lens)
            total, best, lines[key] = left, walk(lens[0], left, n), 0
            for i, length in enumerate(lens, 1):
                chunks, left = chunks - (-length // CHUNK), left - length
                if i < n and lens[i] == length:
                    continue                                      # equals go together
                if 4 * (lens[0] + total - left) < (5 if i < n else 4) * enough:
                    continue
                cost = start + chunk * cols * chunks + (15.0 + walk(lens[i], left, n - i) if i < n else 0.0)
                if cost < best:
                    best, lines[key] = cost, length
        return lines[key]

    def _lengths_and_lines(self, ctx):
        """(a step's lengths, the longest first, what was found out about them), kept with the step: every layer asks. None
        if the step does not say its lengths."""
        host = getattr(ctx, "host", None)
        if host is None or "seq_qstart" not in host:
            return None
        if "chunks_from" not in host:
            host["chunks_from"] = (sorted(self._portion_lengths(ctx).tolist(), reverse=True), {})
        return host["chunks_from"]

    def _delta_in_chunks(self, ctx, N, D, H, Dv):
        """The same for the gated delta rule, whose chunk costs more and whose walk is faster. Measured in us, walk -> chunks, 20
        heads of 128 x 128: 1,000 tokens 238 -> 133, 2 sequences of 500 149 -> 132, 3 of 500 148 -> 157, of 1,000 281 -> 286, 8 of
        1,000 557 -> 707; 32 heads: 256 tokens 76 -> 69, 3 of 1,000 359 -> 412, 8 of 1,000 791 -> 1,068; 8 heads: 3 of 1,000
        241 -> 142, 8 of 1,000 309 -> 287; 10 of 128 x 256: 3 of 1,000 284 -> 238, 8 of 1,000 561 -> 639; 40 of 64 x 64: 256
        65 -> 44, 3 of 1,000 243 -> 237, 8 of 1,000 441 -> 627; 16 of 64 x 128: 8 of 1,000 310 -> 305. 20 heads, 300 tokens beside 60
        decoding rows that walk 93 -> 116, 1,000 256 -> 187."""
        cols = H * -(-Dv // 16)
        if self._lengths_and_lines(ctx) is None and N * cols >= 600 * (ctx.max_q_len - 165):
            return 0
        wide = D / 128.0
        return self._chunks_from(ctx, D, cols, least=self.delta_scan_from, token=0.171 + 0.058 * wide, serial=0.088 + 0.042 * wide,
                                 busy=(2.2 + 1.04 * wide) * 1e-4, start=36.0, chunk=0.02 + 0.012 * wide)

    def _split(self, ctx, least):
        """(most sequences that go in chunks, whether others walk) of a step taken in chunks from ``least`` tokens on."""
        step = None if least <= 1 else self._lengths_and_lines(ctx)
        if step is None:
            return ctx.n_seqs, False
        lens, lines = step
        if least not in lines:
            n_long = sum(n >= least for n in lens)
            lines[least] = n_long, n_long < ctx.n_seqs
        return lines[least]

    def _scan_scratch(self, ctx, N, n_long, sizes):
        """(chunks of the longest portion, chunks of every sequence that one launch takes, whether those lie one behind the
        other, slots, the scratch of ``sizes`` floats per slot, the addresses of its parts): all chunks at once where the scratch allows
        it, else rounds over a few chunks of every sequence with the state in the row between them. ``n_long``: sequences."""
        chunks, per_slot = -(-ctx.max_q_len // CHUNK), 4 * sum(sizes)
        slots, count = N // CHUNK + n_long, chunks
        compact = slots * per_slot <= self.scan_scratch and slots <= 65535
        if not compact:
            count = max(1, min(chunks, self.scan_scratch // (n_long * per_slot), 65535 // n_long))
            slots = n_long * count
        # one allocation, each part on 16 bytes
        at, ends = 0, []
        for n in sizes:
            ends.append(at)
            at += (slots * n + 3) & ~3
        scratch = torch.empty(at, dtype=torch.float32, device=self.device)
        base = scratch.data_ptr()
        return chunks, count, compact, slots, scratch, [c_void_p(base + 4 * e) for e in ends]

    def _scan(self, mode, q, ldq, hq, k, ldk, hk, v, ldv, hv, decay, H, D, Dv, state, stride, offset, ctx, N, out, least, group=1,
              q_f32=True, v_act=False, ones=0, lda=0, params=()):
        """The sequences of ``least`` tokens and more; returns whether others are left to walk. ``q``, ``k``, ``v``, ``decay`` and
        ``params`` are addresses (``c_void_p``), ld* elements from one token to the next, h* from one head to the next."""
        dk = 64 if D <= 64 else 128
        rows = CHUNK * dk if mode in (CHANNEL, BONUS) else CHUNK
        n_long, others = self._split(ctx, least)
        chunks, count, compact, slots, scratch, parts = self._scan_scratch(ctx, N, n_long, [H * _tiles(D, Dv), H * rows, H * dk])
        p = list(params) + [None] * (3 - len(params))
        self.forms["scan"] += 1
        for first in range(0, chunks, count):
            _check(self._scan_lib().soc_scan(
                c_int(mode), q, c_longlong(ldq), c_int(hq), k, c_longlong(ldk), c_int(hk), c_int(group), c_int(1 if q_f32 else 0),
                v, c_longlong(ldv), c_int(hv), c_int(1 if v_act else 0), c_int(ones), decay, c_longlong(lda), *p, c_int(H), c_int(D),
                c_int(Dv), _ptr(state), stride, c_int(offset), _ptr(ctx.seq_qstart), _ptr(ctx.seq_rows), c_int(ctx.n_seqs),
                c_int(least), c_int(n_long), c_int(slots), c_int(first), c_int(count), c_int(1 if compact else 0), _ptr(out),
                *parts, c_int(self.code), self._stream()), "scan")
        return others

    def _delta_scan(self, qk, v, gates, G, H, D, Dv, Dp, state, stride, offset, ctx, N, out, least=1):
        """The gated delta rule in chunks for the sequences of ``least`` tokens and more, from what ``soc_delta_prepare`` leaves."""
        n_long, _ = self._split(ctx, least)
        chunks, count, compact, slots, scratch, parts = self._scan_scratch(ctx, N, n_long, [H * _tiles(D, Dv), H * CHUNK * Dp, H * Dp * Dp])
        self.forms["scan"] += 1
        for first in range(0, chunks, count):
            _check(self._scan_lib().soc_delta_scan(
                _ptr(qk), _ptr(v), _ptr(gates), c_int(G), c_int(H), c_int(D), c_int(Dv), c_int(Dp), _ptr(state), stride, c_int(offset),
                _ptr(ctx.seq_qstart), _ptr(ctx.seq_rows), c_int(ctx.n_seqs), c_int(least), c_int(n_long), c_int(slots), c_int(first),
                c_int(count), c_int(1 if compact else 0), _ptr(out), *parts, c_int(self.code), self._stream()), "delta_scan")
        return out
