"""torch-facing wrappers over ``libjf_layers.so`` (include/jf_layers.h): torch allocates and owns the memory, every operation
runs in the HIP library.  Shapes are checked here, on the host, before a launch.

A step's tokens form one ragged batch (``RaggedBatch``): N token rows, the rows of a request consecutive, with the per-request
records and tiles the kernels read."""
from __future__ import annotations

import bisect
import ctypes as C
import itertools
import math
import operator
import os
import threading
from collections import deque
from dataclasses import dataclass, field
from typing import List, Optional, Sequence, Tuple

import numpy as np
import torch
import torch.nn.functional as F
from torch.autograd import forward_ad
from torch.compiler import is_dynamo_compiling
from torch.utils._device import DeviceContext

from . import _native as N


ATTN_SPLIT_BELOW_TILES, ATTN_SPLIT_WORKGROUPS = 128, 512     # attention: split a tile's keys while tiles x splits stays below ~2 per CU
ATTN_MAX_HEADS_ONE_LAUNCH, ATTN_MAX_VALUE_WIDTH = 16, 128   # what the matrix-core attention kernel takes in one workgroup
# mixed heads: workgroups of 4 wavefronts to aim at (of one: three times as many); scratch at most (1 GiB: more tiles than it holds take turns), as long as it holds a tile's.  us, 8 heads
# over 2 of 128 under a window of 1024, for 512 / 640 / 1024: 777 + 300 tokens beside 30 single ones 105 / 79 / 81, one portion of 1000 54 / 56 / 65.  The form costs a product with the
# values per value head, and is taken for up to 8 of them: us, two sweeps / this, 4 x 2048 tokens, 32 single ones: 8 heads over 1 688 / 102, 122 / 29; 4 over 4 1011 / 179, 196 / 81; 16 over 4
# 1891 / 585, 299 / 93; sizes that went to float multiply-adds before: 12 over 6 51800 / 689, 16 over 8 70400 / 1270
TALK_WORKGROUPS, TALK_SCRATCH_FLOATS = 640, 256 << 20
# attention of a few tokens per request (and of portions too few for the 128-row tiles): workgroups to aim at when keys are shared out, keys of a share at least, and keys up to which they never are: one
# launch and no scratch.  A workgroup has eight wavefronts, so one per CU has every CU's loads on their way; more only add sums to join.  us, workgroups 256 / 512: 32 tokens at 2048, 16 heads of 128 over 4
# 31 / 34, latent of 512 30 / 30, of 256 (48 at 1000) 17 / 23, 8 mixed heads over 2 18 / 18, 16 over 4 29 / 37; 200 tokens at 1000, 16 heads over 4 21 / 29.  Keys of a share 64 / 96 / 128 / 256: one token at 700, 8 heads over
# 2 9.5 / 9.5 / 9.8 / 11.2, mixed 13.2 / 13.4 / 14.0 / 17.8; 32 tokens at 150 9.2 / 9.5 / 9.5 / 7.9
NARROW_WORKGROUPS, TOKEN_KEYS, NARROW_WHOLE = 256, 96, 128
BLOCK_WORKGROUPS = 512               # a draft block's attention without key groups: workgroups to aim at when keys are shared out
SWEEP_SPLIT_BELOW_GROUPS, SWEEP_SPLIT_WORKGROUPS = 512, 2048   # one-sweep attention: its workgroups are small (4 wavefronts, <= 32 rows)
SWEEP_WIDE_ROWS_PER_REQUEST = 16   # one-sweep attention: from this many tokens per request on average a step takes the 128-row tiles
RETENTION_PIECES_FROM, RETENTION_WORKGROUPS = 8, 512     # retention: portions from this many tokens on (retention_pieces_from) run in pieces on the matrix cores; workgroups to aim at (us at 256 / 512: 8 heads of 128, 4 x 2048 tokens 126 / 117, of 64 78 / 70; one of 1000 47 / 47)
RETENTION_CHUNK = 64          # tokens per chunk when a long portion's recurrence is cut into chunks that run side by side
SCAN_PIECES_FROM, SCAN_WAVES = 32, 2048     # linear recurrence: portions from this many tokens on run in pieces on the matrix cores; wavefronts of 32 columns to aim at (us at
                                            # 1024 / 2048 / 4096: 4 x 2048 tokens of 16 heads of 128 141 / 125 / 151, one of 8192 144 / 127 / 156; 2 x 2048 of 8 heads 59 / 63 / 63, 5 x 1500 of 6 heads of 64 44 / 44 / 44)
DELTA_COLUMNS_FROM = 32       # delta rule: from this many tokens in a request's portion on, the state's columns are shared out over wavefronts
DELTA_CHUNKS_FROM = 64        # ... from here on its chunks of 64 tokens go to the matrix instructions (alone in its step; else delta_chunks_from.  us at 16 heads of 128, chunks / columns: 32 tokens 35 / 26, 40 35 / 31, 64 37 / 45, 8 x 64 49 / 67)
DELTA_SCRATCH_FLOATS = 256 << 20     # scratch of those chunks at most (1 GiB: more heads than it holds take turns), as long as it holds one key head's


def _ptr(t: Optional[torch.Tensor]):
    return None if t is None else t.data_ptr()


def _stream(device: torch.device):
    """The current stream's handle (the raw one: no stream object is made for every launch)."""
    if device.type != "cuda":
        return None
    return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device() if device.index is None else device.index)


def _code(dt: torch.dtype) -> int:
    if dt == torch.float32:
        return N.JL_F32
    if dt == torch.bfloat16:
        return N.JL_BF16
    raise ValueError(f"activations must be float32 or bfloat16, got {dt}")


def _need(cond: bool, msg: str) -> None:
    if not cond:
        raise ValueError(msg)


def _dev(t: torch.Tensor) -> None:
    if not t.is_cuda:
        raise N.NativeLibraryError("the layer kernels run on the GPU only (no CPU fallback)")


_H = None                                            # the wrappers' host side in native code: what it does not take comes back as NotImplemented, and the wrapper goes on


def _host():
    global _H
    if _H is None:
        _H = N.host(LINEAR_SMALL_ROWS, LINEAR_ONE_TILE, LINEAR_X_BYTES)
    return _H


_UPLOADS: dict = {}                                  # device index -> the stream its tables are copied on, and a block of its pool
_GONE: dict = {}                                     # a stream's id -> _Gone
GONE_AT_ONCE = 64                                    # tables (of some KB each; built keys' rows of a long step up to a MB) that wait for an event together


class _Gone:
    """Tables uploaded from one stream whose batch is gone.  They are let go, GONE_AT_ONCE at a time, once the stream is done with what lies in front of an upload behind their batch's end.  One
    event says so for all of them: an event takes the host 15 to 20 us (one portion of 200 tokens, us a pass: one per table or per upload 695, this 665, tables on the kernels' stream 655)."""

    def __init__(self, stream: torch.cuda.Stream):
        self.stream, self.tables, self.waiting, self.lock = stream, deque(), deque(), threading.Lock()

    def sweep(self) -> None:
        if len(self.tables) < GONE_AT_ONCE:
            return
        with self.lock:
            while self.waiting and self.waiting[0][0].query():
                for t in self.waiting.popleft()[1]:
                    if torch._C._storage_Use_Count(t.untyped_storage()._cdata) > 2:      # more than this tensor and its storage's object: somebody kept a part of the tables
                        t.record_stream(self.stream)
            left = []
            while self.tables:
                left.append(self.tables.popleft())
            event = torch.cuda.Event()
            event.record(self.stream)
            self.waiting.append((event, left))


def _upload(host, device, held: list) -> torch.Tensor:
    """``host`` on ``device``, there for every stream when this returns.  A copy from ordinary host memory waits for its stream: on one of its own it waits for itself and not for the kernels
    queued so far.  That shows where passes queue behind one another (us a pass, tables on the kernels' stream / on this one: 32 decoding requests of Mikipel 860 / 796, 4 prompts of 2048 of Lokizen
    2402 / 2301).
    The tensor joins ``held``, the batch's list.  Its memory goes back to the copies' stream once the stream that asked for it is done with what lies in front of its first upload behind the batch's
    end: what a caller makes that stream wait for until then (kernels of another stream that read the tables) comes first, as it did when the memory was that stream's own."""
    device = torch.device(device)
    t = torch.from_numpy(host) if isinstance(host, np.ndarray) else host
    if device.type != "cuda":
        return t.to(device)
    if torch.cuda.is_current_stream_capturing():
        raise RuntimeError("a step's tables cannot be copied while a graph is captured")
    here = torch.cuda.current_device()
    index = here if device.index is None else device.index
    if index not in _UPLOADS:
        side = torch.cuda.Stream(index)
        with torch.cuda.stream(side):                    # a block that stays keeps the pool's first segment (2 MB) from being given back and asked for again
            _UPLOADS.setdefault(index, (side, torch.empty(1, dtype=torch.int32, device=device)))
    side, user = _UPLOADS[index][0], torch._C._cuda_getCurrentStream(index)      # (the stream's id, not an object for every upload)
    if user not in _GONE:
        _GONE.setdefault(user, _Gone(torch.cuda.current_stream(index)))
    gone = _GONE[user]
    gone.sweep()
    if index == here:                                    # a fifth of what the context below takes
        torch._C._cuda_setStream(stream_id=side.stream_id, device_index=side.device_index, device_type=side.device_type)
        try:
            up = t.to(device)
        finally:
            torch._C._cuda_setStream(stream_id=user[0], device_index=user[1], device_type=user[2])
    else:
        with torch.cuda.stream(side):
            up = t.to(device)
    held.append((gone.tables, up))
    return up


@dataclass
class RaggedBatch:
    """What one step runs: requests b = 0..B-1 with ``counts[b]`` new tokens from position ``starts[b]``, state slot ``slots[b]``
    and pages ``block_tables[b]``.  Device tensors: ``seq`` [B, 4] int32 {row0, count, pos0, slot}, ``kv_slot`` [N] int64 (pool
    token of every new row), ``tables`` [B, C] int32, ``row_req`` / ``pos`` [N] int32 (request and position of every row).  They are there for every stream when ``build`` returns; a stream
    other than the one that was current then may read them for as long as that one is made to wait for it before it builds its next batch."""
    B: int
    N: int
    counts: List[int]
    starts: List[int]
    seq: torch.Tensor
    kv_slot: torch.Tensor
    tables: torch.Tensor
    row_req: torch.Tensor
    pos: torch.Tensor
    page_size: int
    max_pos: int
    max_page: int
    max_slot: int
    slots: List[int]
    _tiles: dict
    _host_tables: Optional[np.ndarray] = None         # tables on the host, for key_rows and part (None: read back when they need it)
    # the largest portion, and where a tile per request lies in the upload, and behind it, for portions of SCAN_PIECES_FROM tokens on (else 0), a piece per request and the requests' records of them
    _whole: Optional[Tuple[int, torch.Tensor, int, int]] = None      # (None: a request without tokens)
    _held: list = field(default_factory=list, repr=False, compare=False)      # what was uploaded for it, with the list it joins behind the batch's end

    def __del__(self):
        for gone, t in self.__dict__.get("_held", ()):
            gone.append(t)

    @classmethod
    def build(cls, counts: Sequence[int], starts: Sequence[int], slots: Sequence[int], block_tables: Sequence[Sequence[int]],
              page_size: int, device) -> "RaggedBatch":
        if _H is not None or torch.device(device).type == "cuda":
            r = (_H or _host()).step_tables(counts, starts, slots, block_tables, page_size, SCAN_PIECES_FROM)
            if r is not NotImplemented:                  # (us, 32 decoding requests of 33 pages each / one: so 10 / 5, below 40 / 13)
                host, N_, C_, a_seq, a_bt, a_req, a_pos, a_whole, pieced, max_pos, max_page, max_slot, longest, least = r
                B, held_by = len(counts), []
                up = _upload(host, device, held_by)
                words, seq, kv_slot, tables, row_req, pos = _H.step_views(up, B, N_, C_, a_seq, a_bt, a_req, a_pos)
                return cls(B=B, N=N_, counts=list(counts), starts=list(starts), seq=seq, kv_slot=kv_slot, tables=tables, row_req=row_req, pos=pos, page_size=page_size, max_pos=max_pos, max_page=max_page,
                           max_slot=max_slot, slots=list(slots), _tiles={}, _host_tables=host.numpy().view(np.int32)[a_bt:a_bt + B * C_].reshape(B, C_),
                           _whole=(longest, words, a_whole, pieced) if least > 0 else None, _held=held_by)
        B = len(counts)
        if len(starts) != B or len(slots) != B:
            raise ValueError(f"{B} requests, {len(starts)} starts, {len(slots)} slots")
        held = list(map(len, block_tables))              # pages of each request (tables of more requests count in the tables' width alone)
        C_, block_tables, held = max(1, max(held)), block_tables[:B], held[:B]
        for b in range(B):
            if counts[b] and (starts[b] + counts[b] + page_size - 1) // page_size > held[b]:
                raise ValueError(f"request {b}: {held[b]} pages do not hold {starts[b] + counts[b]} tokens")
        counts, starts, slots = list(map(int, counts)), list(map(operator.index, starts)), list(map(int, slots))
        if min(counts) < 0:
            raise ValueError("a request of fewer than no tokens")
        row0 = list(itertools.accumulate(counts, initial=0))
        N_ = row0[B]
        # one upload: the pool tokens (64 bits), then the 32-bit tables, each from a 16-byte border on; `whole`: tiles() and pieces() of steps whose requests are one tile, one piece each (on
        # an idle stream a second upload costs a step of 40 tokens 25 us)
        seq = [x for r in zip(row0, counts, starts, slots) for x in r]
        whole = [x for r in zip(range(B), starts, counts, row0) for x in r]
        longest, pieced = max(counts), 0
        if longest >= SCAN_PIECES_FROM and min(counts) > 0:
            pieced = 4 * B
            whole += [x for r, c, sl in zip(row0, counts, slots) for x in (r, c, sl, 1)]
            whole += [x for b, s, sl in zip(range(B), starts, slots) for x in (b, 1, s, sl)]
        sizes = (4 * B, B * C_, N_, N_, 4 * B, pieced, pieced)
        at = list(itertools.accumulate(((n + 3) // 4 * 4 for n in sizes), initial=2 * (N_ + N_ % 2)))
        host = np.empty(at[-1] // 2, dtype=np.int64)
        words = host.view(np.int32)
        a_seq, a_bt, a_req, a_pos, a_whole = at[:5]
        words[a_seq:a_seq + 4 * B], words[a_whole:a_whole + 4 * B + 2 * pieced] = seq, whole
        bt = words[a_bt:a_bt + B * C_].reshape(B, C_)
        pages = np.fromiter(itertools.chain.from_iterable(block_tables), dtype=np.int64, count=sum(held))
        if min(held) == C_:
            bt[:] = pages.reshape(B, C_)
        else:
            bt[:] = -1
            bt[np.arange(C_) < np.asarray(held)[:, None]] = pages
        if N_ == B and min(counts) == 1:                 # decoding: a row per request
            words[a_req:a_req + N_], words[a_pos:a_pos + N_] = range(B), starts
            host[:N_] = [int(t[s // page_size]) * page_size + s % page_size for t, s in zip(block_tables, starts)]
        elif N_:
            if B == 1:
                rows, pos, first = 0, np.arange(starts[0], starts[0] + N_), 0
            else:
                rows = np.repeat(np.arange(B), counts)
                pos = np.arange(N_) + np.asarray(starts)[rows] - np.asarray(row0)[rows]
                first = np.asarray(list(itertools.accumulate(held, initial=0)))[rows]
            page = pos // page_size
            words[a_req:a_req + N_], words[a_pos:a_pos + N_] = rows, pos
            host[:N_] = pages[first + page] * page_size + (pos - page * page_size)
        held_by = []
        up = _upload(host, device, held_by)
        w32 = up.view(torch.int32)
        return cls(B=B, N=N_, counts=counts, starts=starts, seq=w32.as_strided((B, 4), (4, 1), a_seq), kv_slot=up[:N_], tables=w32.as_strided((B, C_), (C_, 1), a_bt),
                   row_req=w32[a_req:a_req + N_], pos=w32[a_pos:a_pos + N_], page_size=int(page_size),
                   max_pos=max(s + c for s, c in zip(starts, counts)), max_page=int(bt.max()), max_slot=max(slots), slots=slots, _tiles={}, _host_tables=bt,
                   _whole=(longest, w32, a_whole, pieced) if min(counts) > 0 else None, _held=held_by)

    def chunks(self, size: int):
        """A portion of at least two chunks is cut into chunks of ``size`` tokens that the recurrent layers run side by side.
        None when no request of the step is that long.  Else (chunk records [chunks, 4] int32 {row0, count, pos0, chunk index},
        chunk lengths [chunks] int32, request records [B, 4] int32 {first chunk, chunks, pos0, slot})."""
        key = ("chunks", size)
        if key not in self._tiles:
            plan = None
            if max(self.counts) >= 2 * size:
                seq = self.seq.cpu().numpy()
                rec, req = [], []
                for b, (c, s) in enumerate(zip(self.counts, self.starts)):
                    req.append((len(rec), -(-c // size), s, int(seq[b, 3])))
                    for o in range(0, c, size):
                        rec.append((int(seq[b, 0]) + o, min(size, c - o), s + o, len(rec)))
                dev = self.seq.device
                rec = np.asarray(rec, dtype=np.int32).reshape(-1, 4)
                plan = tuple(_upload(t, dev, self._held) for t in (rec, np.ascontiguousarray(rec[:, 1]), np.asarray(req, dtype=np.int32).reshape(-1, 4)))
            self._tiles[key] = plan
        return self._tiles[key]

    def pieces(self, size: int):
        """Every request's portion cut into pieces of ``size`` tokens: (piece records [pieces, 4] int32 {row0, count, slot, 1 for a request's
        last piece}, request records [requests with tokens, 4] int32 {first piece, pieces, pos0, slot}), on the device.  A request without tokens has
        no record: more pieces than records means that some request has several."""
        key = ("pieces", size)
        if key not in self._tiles and self._whole is not None and self._whole[0] <= size and self._whole[3]:
            _, words, at, n = self._whole                # came with the batch's own upload
            self._tiles[key] = tuple(words.as_strided((self.B, 4), (4, 1), at + x * n) for x in (1, 2))
        if key not in self._tiles:
            rec, req, r0 = [], [], 0
            for c, s, sl in zip(self.counts, self.starts, self.slots):
                if c == 0:
                    continue
                req.append((len(rec), -(-c // size), s, sl))
                rec += [(r0 + o, min(size, c - o), sl, int(o + size >= c)) for o in range(0, c, size)]
                r0 += c
            both = _upload(np.asarray(rec + req, dtype=np.int32).reshape(-1, 4), self.seq.device, self._held)
            self._tiles[key] = (both[:len(rec)], both[len(rec):])
        return self._tiles[key]

    def long_pieces(self, size: int, least: int):
        """``pieces`` of the requests with at least ``least`` tokens alone (request records of those), the other requests' rows of ``seq`` and their longest portion (0: none)."""
        key = ("long", size, least)
        if key not in self._tiles:
            rec, req, rest, r0 = [], [], [], 0
            for c, s, sl in zip(self.counts, self.starts, self.slots):
                if c >= least:
                    req.append((len(rec), -(-c // size), s, sl))
                    rec += [(r0 + o, min(size, c - o), sl, int(o + size >= c)) for o in range(0, c, size)]
                else:
                    rest.append((r0, c, s, sl))
                r0 += c
            every = _upload(np.asarray(rec + req + rest, dtype=np.int32).reshape(-1, 4), self.seq.device, self._held)
            self._tiles[key] = (every[:len(rec)], every[len(rec):len(rec) + len(req)], every[len(rec) + len(req):], max((r[1] for r in rest), default=0))
        return self._tiles[key]

    def _pages(self) -> np.ndarray:
        if self._host_tables is None:
            self._host_tables = self.tables.cpu().numpy()
        return self._host_tables

    def key_rows(self, requests: Sequence[int], window: int):
        """The pool tokens that ``requests`` read under ``window`` (0: all before them), request by request in order of position: (tokens [K] int64,
        base [B] int32 with the place of request b's position j at base[b] + j)."""
        key = ("keys", tuple(requests), window)
        if key not in self._tiles:
            # page by page, tokens and bases in one upload, which small steps wait for (us of the host, token by token / page by page: 8 requests of 120 keys 54 / 34, 64 of 150
            # 375 / 200, 4 of 2048 88 / 36, and 25 per upload)
            size, at = self.page_size, 0
            pages, within = self._pages().astype(np.int64) * size, np.arange(size, dtype=np.int64)
            spans = [(b, max(0, self.starts[b] - window + 1) if window > 0 else 0, self.starts[b] + self.counts[b]) for b in requests]
            total = sum(end - first for _, first, end in spans)
            host = np.zeros(total + (self.B + 1) // 2, dtype=np.int64)               # the tokens, then the bases as 32-bit numbers
            base = host[total:].view(np.int32)
            for b, first, end in spans:
                p0 = first // size
                host[at:at + end - first] = (pages[b, p0:(end - 1) // size + 1, None] + within).ravel()[first - p0 * size:end - p0 * size]
                base[b] = at - first
                at += end - first
            up = _upload(host, self.seq.device, self._held)
            self._tiles[key] = (up[:total], up[total:].view(torch.int32)[:self.B])
        return self._tiles[key]

    def part(self, requests: Sequence[int]):
        """``requests`` as a batch of their own and the rows of this batch that are theirs ([n] int64)."""
        key = ("part", tuple(requests))
        if key not in self._tiles:
            row0 = np.concatenate([[0], np.cumsum(self.counts)])
            rows = np.concatenate([np.arange(row0[b], row0[b + 1], dtype=np.int64) for b in requests])
            sub = RaggedBatch.build([self.counts[b] for b in requests], [self.starts[b] for b in requests], [self.slots[b] for b in requests],
                                    [self._pages()[b] for b in requests], self.page_size, self.seq.device)
            self._tiles[key] = (sub, _upload(rows, self.seq.device, self._held))
        return self._tiles[key]

    def tiles(self, tq: int, longest_first: bool = False, requests: Optional[Sequence[int]] = None) -> torch.Tensor:
        """[n_tiles, 4] int32 {b, first query position, count, first row}: each request's rows cut into runs of at most ``tq``; with
        ``longest_first`` those with the most positions in front of them come first; only those of ``requests`` when given."""
        key = ("longest first" if longest_first else "in order", tq, None if requests is None else tuple(requests)) if longest_first or requests is not None else tq
        t = self._tiles.get(key)
        if t is None and key == tq and self._whole is not None and self._whole[0] <= tq:
            t = self._tiles[key] = self._whole[1].as_strided((self.B, 4), (4, 1), self._whole[2])      # came with the batch's own upload
        if t is None and _H is not None and requests is None:
            rows = _H.tile_records(self.counts, self.starts, tq, longest_first)
            if rows is not NotImplemented:
                t = self._tiles[key] = _upload(rows, self.seq.device, self._held)
        if t is None:
            rows, r0 = [], 0
            for b, (c, s) in enumerate(zip(self.counts, self.starts)):
                for o in range(0, c if requests is None or b in requests else 0, tq):
                    rows.append((b, s + o, min(tq, c - o), r0 + o))
                r0 += c
            if longest_first:
                rows.sort(key=lambda r: -r[1])
            t = self._tiles[key] = _upload(np.asarray(rows, dtype=np.int32).reshape(-1, 4), self.seq.device, self._held)
        return t


LINEAR_SMALL_ROWS, LINEAR_ONE_TILE = 64, 4096       # jl_linear_small: rows at most; W's rows up to which a workgroup takes 16 of them
LINEAR_X_BYTES = 128 << 10           # ... and the bytes of x that a CU reads up to which it is the faster one
_LINEAR_SAME, _LINEAR_FLOAT, _LINEAR_ROUNDED_FLOAT = 0, 1, 2
_LINEAR_TYPES = (torch.bfloat16, torch.float32)


def linear_small(n: int, k: int, o: int, itemsize: int) -> bool:
    """Whether ``linear`` takes n rows of k values times [o, k] to the package's launch.  Every workgroup reads all rows of x: 16 of W's rows each up to LINEAR_ONE_TILE, then 32 and 64.
    us of GPU time, own / library, at the line (bfloat16): 32 rows of 2048 by 2048 8.3 / 8.5, by 5120 12.8 / 12.4, 64 rows of 1024 by 4096 8.1 / 8.7; beyond it: 32 rows of 4096 by
    2048 15.4 / 12.3, 64 rows of 2048 by 2048 12.1 / 9.2, 32 rows of 2048 by 32000 36.8 / 31.1.  float: 16 rows of 2048 by 2048 11.9 / 12.1; beyond, 32 rows 17.5 / 12.5."""
    tile = 16 if o <= LINEAR_ONE_TILE or n == 1 else 32 if o <= 4 * LINEAR_ONE_TILE else 64
    return 0 < n <= LINEAR_SMALL_ROWS and n * k * itemsize * -(-o // (tile * 256)) <= LINEAR_X_BYTES


def linear_mid(n: int, k: int, o: int, dtype: torch.dtype) -> int:
    """Whether ``linear`` takes n rows of k values times [o, k] to the launch for some hundred to a few thousand bfloat16 rows.  2 (under autocast as well), for any number of rows: up to 512 tiles of 64 x 64
    where k is up to 1024, up to 256 where it is up to 2048.  1, up to 2304 rows and w of up to 64 MB: k up to 2048 and up to 256 tiles of 128 x 128 (k up to 1024: two of those per CU, 512); k up to 4096
    from 300 rows on with 80 to 256 tiles of 64 x 64.  There its GPU time is about the library's and the call costs 16 us less of the host, which steps of up to some thousand tokens wait for (a block of four
    layers of 896 wide by 256 tokens 557 -> 354 us).  us of GPU time, operands from memory, library / own: 300 rows of 512 by 6144 12.1 / 9.8, 1500 of 1536 by 1024 13.2 / 12.1, 1024 of 2048 by 4096 25.2 /
    24.2, 2048 of 2048 by 2048 24.4 / 24.3, 300 of 4096 by 2048 21.6 / 20.1; two tiles per CU 2048 of 512 by 3072 15.2 / 13.3, of 1024 by 3072 18.4 / 19.1, at worst 1024 of 1024 by 6144 19.2 / 23.9.  Beyond
    the line: deeper ones of two per CU, 700 of 2048 by 6144 26.8 / 33.3, 2048 of 1536 by 3072 24.6 / 32.8 (safisun's 700 tokens of 2048 wide 875 -> 813 us a pass with those at the library); of 6 and 8 KB
    many tiles, 700 of 4096 by 2048 25.5 / 31.4, and few, which the library shares out, 512 of 4096 by 512 11.0 / 17.6; more rows, 3000 of 2048 by 512 14.7 / 17.0, 4096 of 1024 by 1024 13.9 / 14.5; w that
    takes longer to read than to multiply, 256 of 2048 by 32000 45.3 / 52.4."""
    return int(N.layers().jl_linear_mid_ok(n, k, o)) if dtype == torch.bfloat16 else 0


def linear_split(n: int, k: int, o: int) -> bool:
    """Whether ``linear`` takes n float rows of k values times [o, k] to the bfloat16 matrix instructions in three terms per operand: where their tiles fill the chip well enough (the rule and its
    figures are the launch's, jl_linear_split_ok)."""
    return bool(N.layers().jl_linear_split_ok(n, k, o))


def _plain(*tensors: Optional[torch.Tensor]) -> bool:
    """Whether a launch on these tensors' memory is all that a library's call on them would be: no subclass (fake tensors among them), transform's wrapper, lazy form, sparse layout or forward-mode
    tangent, no trace that records calls, and no mode that is to see the call (one that only names a default device has nothing to see)."""
    modes = torch.overrides._get_current_function_mode_stack() if torch._C._len_torch_function_stack() else ()
    if torch._C._get_tracing_state() is not None or torch._C._len_torch_dispatch_stack() or any(type(m) is not DeviceContext for m in modes):
        return False
    dual = forward_ad._current_level >= 0
    return all(t is None or (type(t) in (torch.Tensor, torch.nn.Parameter) and t.layout == torch.strided and not torch._C._functorch.is_functorch_wrapped_tensor(t) and not t.is_neg() and
                             not t._is_zerotensor() and not (dual and forward_ad.unpack_dual(t).tangent is not None)) for t in tensors)


def linear(x: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor] = None, float_out: Optional[bool] = None) -> torch.Tensor:
    """x [N, K] times w [O, K] transposed (+ bias [O]): the package's launches for few rows (decoding, ``linear_small``), some hundred to a few thousand (``linear_mid``) and many float ones
    (``linear_split``), the library's product for the others and for what a launch would pass by (``_plain``).  ``float_out`` None: x's dtype; True: the float sums, unrounded; False: float, rounded to x's dtype first.  w (and bias) may be float beside a 16-bit x, which then
    counts as float: give ``float_out`` True.  What the launches do not take (other types, devices that differ, gradients wanted) is the library's to compute or refuse."""
    _dev(x)
    launch = not is_dynamo_compiling()    # (a compiler follows the library's call alone)
    if launch:
        r = (_H or _host()).linear(x, w, bias, float_out)
        if r is not NotImplemented:
            return r
    n, k = x.shape
    o, dt, wt = w.shape[0], x.dtype, w.dtype
    same = wt == dt
    _need(same or (wt == torch.float32 and float_out is True), "linear: w of x's dtype, or float with a float result")
    small = launch and n <= LINEAR_SMALL_ROWS and linear_small(n, k, o, w.element_size())
    split = launch and not small and wt == torch.float32 and linear_split(n, k, o) and not torch.is_autocast_enabled("cuda")
    mid = linear_mid(n, k, o, dt) if launch and same and not small else 0
    if launch and (small or split or mid == 2 or (mid and not torch.is_autocast_enabled("cuda"))) and _plain(x, w, bias):
        size = w.element_size()
        if (w.shape[1] == k and w.is_contiguous() and x.stride(1) == 1 and x.stride(0) >= k and k * size % 16 == 0 and x.stride(0) * x.element_size() % 16 == 0 and
                (x.data_ptr() | w.data_ptr()) % 16 == 0 and (bias is None or (bias.dtype == wt and bias.shape == (o,) and bias.is_contiguous())) and dt in _LINEAR_TYPES and k > 0 and
                w.get_device() == x.get_device() and (bias is None or bias.get_device() == x.get_device()) and
                not (torch.is_grad_enabled() and (x.requires_grad or w.requires_grad or (bias is not None and bias.requires_grad)))):
            mode = _LINEAR_SAME if float_out is None else _LINEAR_FLOAT if float_out else _LINEAR_ROUNDED_FLOAT
            if small:
                out = torch.empty((n, o), dtype=dt if float_out is None else torch.float32, device=x.device)
                N.check_layers(N.layers().jl_linear_small(x.data_ptr(), _code(dt), n, x.stride(0), w.data_ptr(), _code(wt), k, o, _ptr(bias), out.data_ptr(), o, mode,
                                                         _stream(x.device)), "jl_linear_small")
                return out
            if split:
                x = x.float()
                out = torch.empty((n, o), dtype=torch.float32, device=x.device)
                N.check_layers(N.layers().jl_linear_split(x.data_ptr(), n, x.stride(0), w.data_ptr(), k, o, _ptr(bias), out.data_ptr(), o, _stream(x.device)), "jl_linear_split")
                return out
            if n * x.stride(0) * size < 1 << 32:
                out = torch.empty((n, o), dtype=dt if float_out is None else torch.float32, device=x.device)
                N.check_layers(N.layers().jl_linear_mid(x.data_ptr(), _code(dt), n, x.stride(0), w.data_ptr(), k, o, _ptr(bias), out.data_ptr(), o, mode, _stream(x.device)),
                               "jl_linear_mid")
                return out
    # the library's, with as little before it as there was when models called it themselves
    if not same:
        x = x.float()
    if float_out and wt != torch.float32:
        y = torch.mm(x, w.t(), out_dtype=torch.float32)
        return y if bias is None else y + bias
    if float_out and bias is None:
        return torch.mm(x, w.t())
    y = F.linear(x, w, bias)
    return y if float_out is None else y.float()


def linear_add_(out: torch.Tensor, x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """``out`` [N, O] plus x [N, K] times w [O, K] transposed, in place, rounded once: the package's launch (``linear_mid``), or the library's product."""
    if not (is_dynamo_compiling() or (_H or _host()).linear_add(out, x, w) is NotImplemented):
        return out
    return out.addmm_(x, w.t())


def rms_norm(x: torch.Tensor, w: torch.Tensor, eps: float) -> torch.Tensor:
    """x / sqrt(mean(x^2) + eps) * w over the last axis, in x's dtype: the package's launch, or the library's function for what that does not take (other types, gradients, autocast, wide rows)."""
    if x.is_cuda and not is_dynamo_compiling():
        r = (_H or _host()).rms_norm(x, w, eps)
        if r is not NotImplemented:
            return r
    return F.rms_norm(x, (x.shape[-1],), w, eps)


def embed_scale(embed: torch.Tensor, ids: torch.Tensor, scale: float, want_copy: bool,
                out: Optional[torch.Tensor] = None, copy_dtype: torch.dtype = torch.float32) -> Tuple[torch.Tensor, Optional[torch.Tensor]]:
    """Rows ``ids`` of ``embed`` times ``scale`` as float [N, W] (written into ``out`` when given), and a second copy with ``want_copy``
    (float, or rounded to bfloat16 with ``copy_dtype``)."""
    _dev(embed)
    r = (_H or _host()).embed_scale(embed, ids, scale, want_copy, out, copy_dtype)
    if r is not NotImplemented:
        return r
    _need(embed.dim() == 2 and embed.is_contiguous() and ids.dtype == torch.int64 and ids.is_contiguous(), "embed_scale: embed [V, W], ids int64 [N]")
    n, W = ids.numel(), embed.shape[1]
    if out is not None:
        _need(out.dtype == torch.float32 and out.is_contiguous() and tuple(out.shape) == (n, W), "embed_scale: out float [N, W]")
    x = out if out is not None else torch.empty((n, W), dtype=torch.float32, device=embed.device)
    _need(copy_dtype in (torch.float32, torch.bfloat16), "embed_scale: the copy is float or bfloat16")
    x0 = torch.empty((n, W), dtype=copy_dtype, device=embed.device) if want_copy else None
    wide = copy_dtype == torch.float32
    N.check_layers(N.layers().jl_embed_scale(_ptr(embed), _code(embed.dtype), _ptr(ids), n, W, float(scale), _ptr(x), _ptr(x0) if wide else None,
                                            None if wide else _ptr(x0), _stream(embed.device)), "jl_embed_scale")
    return x, x0


def add_rmsnorm(x: torch.Tensor, y: Optional[torch.Tensor], x0: Optional[torch.Tensor], w: Optional[torch.Tensor], eps: float,
                out_dtype: Optional[torch.dtype]) -> Optional[torch.Tensor]:
    """x (float [N, W], in place) += y summed over its middle axis ([N, W] or [N, S, W], float or bf16) + x0; returns
    rms_norm(x) * w in ``out_dtype`` (None: the update only)."""
    _dev(x)
    r = (_H or _host()).add_rmsnorm(x, y, x0, w, eps, out_dtype)
    if r is not NotImplemented:
        return r
    n, W = x.shape
    _need(x.dtype == torch.float32 and x.is_contiguous(), "add_rmsnorm: x must be contiguous float32 [N, W]")
    cnt = 0
    if y is not None:
        _need(y.is_contiguous() and y.shape[0] == n and y.shape[-1] == W and y.dim() in (2, 3), "add_rmsnorm: y must be [N, W] or [N, S, W]")
        cnt = 1 if y.dim() == 2 else y.shape[1]
    if x0 is not None:
        _need(x0.shape == x.shape and x0.dtype == torch.float32 and x0.is_contiguous(), "add_rmsnorm: x0 must match x")
    out = None
    if out_dtype is not None:
        out = torch.empty((n, W), dtype=out_dtype, device=x.device)
        if w is not None:
            _need(w.dtype == out_dtype and w.numel() == W and w.is_contiguous(), "add_rmsnorm: the weight has the output's dtype and W entries")
    N.check_layers(N.layers().jl_add_rmsnorm(_ptr(x), _ptr(y), _code(y.dtype) if y is not None else 0, cnt, _ptr(x0), _ptr(w), float(eps),
                                            _ptr(out), _code(out_dtype or torch.float32), n, W, _stream(x.device)), "jl_add_rmsnorm")
    return out


def qk_norm_append(proj: torch.Tensor, cols: Tuple[int, int, int], H: int, G: int, D: int, Dv: int, wq: torch.Tensor, wk: torch.Tensor,
                   eps: float, k_cache: torch.Tensor, v_cache: torch.Tensor, kv_slot: torch.Tensor, rot_dims: int = 0, pairing: int = N.JL_ROT_HALVES,
                   batch: Optional["RaggedBatch"] = None, cos: Optional[torch.Tensor] = None, sin: Optional[torch.Tensor] = None) -> torch.Tensor:
    """RMS norm of q over all its heads together (and of k over its), with ``rot_dims`` the rotation of both by position behind it (needs
    ``batch`` and its angle tables), keys / values appended to the pools.  Returns q [N, H*D]."""
    _dev(proj)
    r = (_H or _host()).qk_norm_append(proj, *cols, H, G, D, Dv, wq, wk, eps, k_cache, v_cache, kv_slot, rot_dims, pairing, batch.N if batch is not None else 0,
                                       batch.max_pos if batch is not None else 0, batch.pos if batch is not None else None, cos, sin)
    if r is not NotImplemented:
        return r
    n, ld = proj.shape
    dt = proj.dtype
    _need(proj.is_contiguous() and kv_slot.dtype == torch.int64 and kv_slot.numel() == n, "qk_norm_append: proj [N, ld], one pool token per row")
    _need(wq.numel() == H * D and wk.numel() == G * D and wq.dtype == dt and wk.dtype == dt, "qk_norm_append: norm weights over the whole projections")
    _need(k_cache.dtype == dt and v_cache.dtype == dt and k_cache.is_contiguous() and v_cache.is_contiguous() and
          k_cache.shape[-1] == G * D and v_cache.shape[-1] == G * Dv and k_cache.shape[0] == v_cache.shape[0], "qk_norm_append: pools [tokens, G*D] / [tokens, G*Dv]")
    if rot_dims:
        _need(batch is not None and n == batch.N and rot_dims % 2 == 0 and 0 <= rot_dims <= D, "qk_norm_append: the rotation needs the batch and an even number of dimensions up to D")
        _angle_tables(rot_dims, cos, sin, batch, "qk_norm_append")
    q = torch.empty((n, H * D), dtype=dt, device=proj.device)
    N.check_layers(N.layers().jl_qk_norm_append(_ptr(proj), _code(dt), n, ld, cols[0], cols[1], cols[2], H, G, D, Dv, _ptr(wq), _ptr(wk), float(eps),
                                               _ptr(q), _ptr(k_cache), _ptr(v_cache), _ptr(kv_slot), int(rot_dims), int(pairing), _ptr(batch.pos) if rot_dims else None,
                                               _ptr(cos) if rot_dims else None, _ptr(sin) if rot_dims else None, _stream(proj.device)), "jl_qk_norm_append")
    return q


def _check_gate_sink(gate, sink, gate_per_head: bool, n: int, H: int, Dv: int, dt, what: str) -> None:
    if gate is not None:
        _need(gate.shape == (n, H if gate_per_head else H * Dv) and gate.stride(1) == 1 and gate.dtype == dt,
              f"{what}: gate [N, H*Dv], or [N, H] with one gate per head")
    if sink is not None:
        _need(sink.dtype == torch.float32 and sink.is_contiguous() and sink.numel() == H, f"{what}: sink float [H]")


def _attn_out(out: Optional[torch.Tensor], n: int, width: int, dtype: torch.dtype, device, what: str) -> torch.Tensor:
    """The output matrix [n, width]: a new one, or the caller's column range of wider rows."""
    if out is None:
        return torch.empty((n, width), dtype=dtype, device=device)
    _need(tuple(out.shape) == (n, width) and out.dtype == dtype and out.stride(1) == 1, f"{what}: out [N, H*Dv] of the output's dtype, contiguous along a row")
    return out


def _fours(out: torch.Tensor) -> bool:
    """Whether rows of ``out`` can be stored four values at a time."""
    return out.stride(0) % 4 == 0 and out.data_ptr() % (4 * out.element_size()) == 0


def attn_tile_rows(dtype: torch.dtype, H: int, G: int, D: int, Dv: int, k_ld: int = 0, v_ld: int = 0) -> int:
    tq = int(N.layers().jl_attn_tile_rows(_code(dtype), H, G, D, Dv, k_ld, v_ld))
    if tq <= 0:
        raise ValueError(f"attention sizes heads={H} kv_heads={G} dim={D} vdim={Dv} exceed the kernel's tile")
    return tq


def _attn_args(q, k_cache, v_cache, out, batch: RaggedBatch, tiles, gate, sink, rel, lut, talk, scratch, q_pack, scale, softcap, out_scale, H, G, Gv, D, Dv, window, keep_first, chunk, tq, splits,
               out_dtype, gate_heads) -> N.AttnArgs:
    """The arguments of an attention launch whose operands the caller has checked."""
    a, numbers = N.AttnArgs(), (batch.page_size, H, G, Gv, D, Dv, int(window), int(keep_first), int(chunk), tq, splits, out_dtype, int(gate_heads))
    if (_H or _host()).attention_args(C.addressof(a), q, k_cache, v_cache, out, batch.tables, tiles, gate, sink, rel, lut, talk, scratch, q_pack, float(scale), float(softcap), float(out_scale),
                                      *numbers) is not NotImplemented:
        return a
    return N.AttnArgs(q=_ptr(q), k_cache=_ptr(k_cache), v_cache=_ptr(v_cache), out=_ptr(out), block_tables=_ptr(batch.tables), tiles=_ptr(tiles), gate=_ptr(gate),
                      gate_ld=gate.stride(0) if gate is not None else 0, sink=_ptr(sink), rel=_ptr(rel), lut=_ptr(lut), talk=_ptr(talk), scratch=_ptr(scratch), q_pack=_ptr(q_pack),
                      lut_len=(lut.numel() if lut is not None else rel.shape[0]) if rel is not None else 0, scale=float(scale), softcap=float(softcap), out_scale=float(out_scale),
                      bt_stride=batch.tables.shape[1], n_tiles=tiles.shape[0], n_rows=q.shape[0], k_ld=k_cache.stride(0), v_ld=v_cache.stride(0), out_ld=out.stride(0), dtype=_code(q.dtype),
                      **dict(zip(("page_size", "H", "G", "Gv", "D", "Dv", "window", "keep_first", "chunk", "TQ", "splits", "out_dtype", "gate_heads"), numbers)))


def _few(batch: RaggedBatch, heads: int, rows: int, tq: int) -> int:
    """The most queries of a tile of up to ``tq`` where that is at most ``rows`` (query, head) rows, ``heads`` to a query (0: more)."""
    most = tq if batch._whole is None else min(batch._whole[0], tq)
    return most if most * heads <= rows else 0


def _token_latent(H: int, D: int, Dv: int) -> bool:
    """Whether latent rows of D columns, the first Dv of them values, have the sizes of the launches for a few tokens (jl_attn_token.hip) with H heads."""
    return H <= 32 and D <= (Dv + 127) // 128 * 128 + 64


def _token_splits(reach: int, units: int) -> int:
    """Shares of the keys for ``units`` workgroups' worth of rows with up to ``reach`` keys each.  The joining launch has eight shares on their way at once, so more than that from 512 keys a share on
    only (4 tokens at 2000, 16 heads over 1, 8 / 16 / 32 shares 12.4 / 14.8 / 22.7 us)."""
    return max(1, min(-(-reach // TOKEN_KEYS), NARROW_WORKGROUPS // units, max(8, -(-reach // 512)), 64))


def attn_window(q: torch.Tensor, gate: Optional[torch.Tensor], k_cache: torch.Tensor, v_cache: torch.Tensor, batch: RaggedBatch,
                H: int, G: int, D: int, Dv: int, scale: float, window: int, keep_first: int, rel: Optional[torch.Tensor],
                lut: Optional[torch.Tensor], talk: Optional[torch.Tensor], value_heads: int = 0, float_out: bool = False,
                sink: Optional[torch.Tensor] = None, gate_per_head: bool = False, chunk: int = 0, softcap: float = 0.0, out_scale: float = 1.0,
                out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """q [N, H*D]; gate a [N, H*Dv] view (column range of the projection output, row stride free; [N, H] with ``gate_per_head``) or
    None.  ``sink`` float [H]: one more term exp(sink_h) in every softmax denominator of head h.  Returns [N, H*Dv].
    The pools may be column ranges of wider rows (``v_cache`` may be a view into ``k_cache``).  ``value_heads`` (0: G) < G: key head
    c reads value head c % value_heads — several score maps over the same values.  ``float_out``: float outputs from bfloat16
    inputs (for what is subtracted or normalised next).  ``chunk`` > 0: a query sees the keys of its own run of ``chunk`` positions only (no
    window beside it).  ``softcap`` > 0: scores pass softcap * tanh(s / softcap).  ``out_scale`` multiplies the outputs, which go to ``out``
    (a column range of wider rows) when given."""
    _dev(q)
    dt = q.dtype
    n = q.shape[0]
    Gv = value_heads or G
    _need(q.is_contiguous() and q.shape[1] == H * D and n == batch.N, "attn_window: q [N, H*D] of the batch")
    _need(G % Gv == 0 and k_cache.dtype == dt and v_cache.dtype == dt and k_cache.dim() == 2 and v_cache.dim() == 2 and k_cache.shape[1] == G * D and
          v_cache.shape[1] == Gv * Dv and k_cache.stride(1) == 1 and v_cache.stride(1) == 1 and k_cache.shape[0] == v_cache.shape[0],
          "attn_window: pool dtype / widths")
    k_ld, v_ld = k_cache.stride(0), v_cache.stride(0)
    pool_tokens = k_cache.shape[0]
    _need(pool_tokens % batch.page_size == 0 and batch.max_page < pool_tokens // batch.page_size, "attn_window: a page lies outside the pool")
    _check_gate_sink(gate, sink, gate_per_head, n, H, Dv, dt, "attn_window")
    for t, shape in ((rel, None), (talk, (H, H))):
        if t is not None:
            _need(t.dtype == torch.float32 and t.is_contiguous() and (shape is None or tuple(t.shape) == shape), "attn_window: float tables")
    if rel is not None:                                  # rel [rows, H] with lut [positions] -> row, or rel [positions, H] by distance itself
        _need(rel.shape[1] == H and (lut is None or lut.dtype == torch.int32), "attn_window: rel [rows, H] (+ int32 lut)")
    _need(chunk <= 0 or (window <= 0 and keep_first <= 0), "attn_window: chunks exclude a window and kept first tokens")
    out = _attn_out(out, n, H * Dv, torch.float32 if float_out else dt, q.device, "attn_window")
    if (talk is not None and sink is None and chunk <= 0 and softcap <= 0 and Gv == G and N.layers().jl_attn_talk_ok(_code(dt), H, G, D, Dv, k_ld, v_ld) and _fours(out) and
            not (q.data_ptr() | k_cache.data_ptr() | v_cache.data_ptr()) % 16 and not os.environ.get("JL_ATTN_NO_MFMA")):
        few = _few(batch, H, 16, 32 * G // H) if G in (1, 2, 4) and batch._whole is not None and batch._whole[0] * H <= 16 else 0
        wide = not few and n >= SWEEP_WIDE_ROWS_PER_REQUEST * batch.B
        tq = int(N.layers().jl_attn_talk_tile_rows(H, G, int(wide)))
        tiles = batch.tiles(tq, longest_first=wide)
        reach = batch.max_pos if window <= 0 else min(batch.max_pos, int(window) + int(keep_first) + tq)
        if few:
            splits = _token_splits(reach, tiles.shape[0] * -(-G // 2))
        else:
            splits = max(1, min(-(-reach // 64), (TALK_WORKGROUPS if wide else 3 * TALK_WORKGROUPS) // (tiles.shape[0] * G * G), 64))
        per_tile = int(N.layers().jl_attn_talk_scratch_floats(1, tq, H, G, Dv, splits))
        pass_tiles = min(tiles.shape[0], max(1, TALK_SCRATCH_FLOATS // per_tile))
        scratch = torch.empty((per_tile * pass_tiles,), dtype=torch.float32, device=q.device)
        a = _attn_args(q, k_cache, v_cache, out, batch, tiles, gate, None, rel, lut, talk, scratch, None, scale, 0.0, out_scale, H, G, Gv, D, Dv, window, max(0, int(keep_first)), 0, tq, splits,
                       N.JL_OUT_F32 if float_out and dt != torch.float32 else N.JL_OUT_SAME, gate_per_head)
        a.longest = few
        N.check_layers(N.layers().jl_attn_talk(C.byref(a), int(wide), pass_tiles, _stream(q.device)), "jl_attn_talk")
        return out
    tq = attn_tile_rows(dt, H, G, D, Dv, k_ld, v_ld)
    tiles = batch.tiles(tq)
    # few tiles with many keys (decoding): share each tile's keys out over workgroups until the chip is full
    splits, scratch = 1, None
    if tq == 32 and tiles.shape[0] < ATTN_SPLIT_BELOW_TILES:
        reach = min(batch.max_pos, chunk + tq) if chunk > 0 else batch.max_pos if window <= 0 else min(batch.max_pos, int(window) + int(keep_first) + tq)
        splits = max(1, min(-(-reach // 64), ATTN_SPLIT_WORKGROUPS // tiles.shape[0], 64))
        if splits > 1:
            scratch = torch.empty((int(N.layers().jl_attn_scratch_floats(tiles.shape[0], n, H, Dv, splits)),), dtype=torch.float32, device=q.device)
    q_pack = torch.empty((tiles.shape[0] * 32 * H * D,), dtype=dt, device=q.device) if tq == 32 else None
    a = _attn_args(q, k_cache, v_cache, out, batch, tiles, gate, sink, rel, lut, talk, scratch, q_pack, scale, softcap, out_scale, H, G, Gv, D, Dv, window, keep_first, chunk, tq, splits,
                   N.JL_OUT_F32 if float_out and dt != torch.float32 else N.JL_OUT_SAME, gate_per_head)
    N.check_layers(N.layers().jl_attn_window(C.byref(a), _stream(q.device)), "jl_attn_window")
    return out


def attn_block_ok(dtype: torch.dtype, device: torch.device, D: int) -> bool:
    """Whether ``attn_block`` takes heads of D values of this dtype."""
    return device.type == "cuda" and dtype == torch.bfloat16 and bool(N.layers().jl_attn_block_ok(N.JL_BF16, D))


def block_slots(positions: torch.Tensor, T: int, row_prompt: torch.Tensor, row_cand: torch.Tensor, row_len: torch.Tensor, S_max: int, T_max: int, candidates: bool):
    """Cache slots of a draft block's tokens (int64 [R*T], -1: none) and, with ``candidates``, their slots in the candidate scratch (else None); inputs int32."""
    _dev(positions)
    for t in (positions, row_prompt, row_cand, row_len):
        _need(t.dtype == torch.int32 and t.is_contiguous() and t.numel() * (1 if t is positions else T) == positions.numel() and t.get_device() == positions.get_device(),
              "block_slots: contiguous int32 [R*T] positions, [R] rows on one device")
    out = torch.empty((2 if candidates else 1, positions.numel()), dtype=torch.int64, device=positions.device)
    N.check_layers(N.layers().jl_block_slots(positions.data_ptr(), row_prompt.data_ptr(), row_cand.data_ptr(), row_len.data_ptr(), row_len.numel(), T, S_max, T_max, out[0].data_ptr(),
                                             out[1].data_ptr() if candidates else None, _stream(positions.device)), "jl_block_slots")
    return out[0], out[1] if candidates else None


def _block_plan(heads: int, GT: int, max_keys: int, D: int):
    """(shares of the keys, whether a workgroup's wavefronts take keys in groups) for ``heads`` (row, key head) pairs of GT (head, token) rows.  Groups, one workgroup of 64 rows per CU, where
    those fit the chip at once, unless keys are many and few shares of them fit; us with / without, 8 heads of 128 over 2, 32 tokens, context 512: 64 rows (256 workgroups) 20.6 / 27.4,
    96 rows 37.1 / 28.9; context 4000: 24 rows 48.9 / 44.7, 48 rows 76.3 / 61.3; 16 tokens, whose 64 rows leave half of the other form's tiles empty, 64 rows, context 4000: 52.2 / 57.1.  A share more
    costs its sums' way through memory, by the rows, and a launch, which takes the host 3 us: one row, whole / in two, 256 keys 13.2 / 16.2, 512 17.5 / 16.8, heads of 64 512 12.1 / 16.7, 1000
    16.4 / 16.6; context 500 / 1000 / 4000 / 16000: 2, 4, 8 and 16 shares are the fastest; 32 rows, context 512: one 19.0, two 21.6, context 2000: 44.1 and 33.9.  Without groups two workgroups per CU
    as far as a share has 500 keys (750 of up to 64 columns): one share / two / three, 80 rows, context 1000 45.2 / 42.6 / 37.9; one / two, 96 rows 512 27.7 / 32.1, 1000 45.3 / 44.0, 1500 60.9 / 52.3,
    64 rows of 14 heads of 64 over 2 1000 27.1 / 31.0, 2000 48.2 / 43.5."""
    units = heads * -(-GT // 64)
    if units <= 256 and (max_keys <= 2500 or units <= 85 or (units <= 128 and (D <= 64 or 8 * GT < 896 * -(-GT // 128)))):
        if max_keys < (300 if D > 64 else 900) or units > 128 or units == 0:
            return 1, 1
        return min(256 // units, math.isqrt(max_keys // (64 + 2 * units))) or 1, 1
    return max(1, min(BLOCK_WORKGROUPS // (heads * -(-GT // 128)), max_keys // (500 if D > 64 else 750))), 0


def attn_block(q: torch.Tensor, T: int, k: torch.Tensor, v: torch.Tensor, kv_len: torch.Tensor, row_len: torch.Tensor, max_keys: int, row_prompt: Optional[torch.Tensor] = None,
               tables: Optional[torch.Tensor] = None, row_cand: Optional[torch.Tensor] = None, ck: Optional[torch.Tensor] = None, cv: Optional[torch.Tensor] = None,
               scale: Optional[float] = None) -> torch.Tensor:
    """Attention of a draft block: q [R, nkv, G*T, D] over k, v [blocks, nkv, page, D].  Token t of row r sees the row's first kv_len[r] keys and the block's tokens up to
    min(t, row_len[r] - 1), at most ``max_keys`` in all: in cache row row_prompt[r], or in the blocks tables[r] lists; with ``ck`` / ``cv`` [rows, nkv, T_max, D], rows whose row_cand is
    not negative have the block's keys there.  Integers int32.  Returns [R*T, nkv*G*D]."""
    _dev(q)
    R, nkv, GT, D = q.shape
    G = GT // T
    for t in (q, k, v) + ((ck, cv) if ck is not None else ()):
        _need(t.is_contiguous() and t.dtype == torch.bfloat16 and t.dim() == 4 and t.shape[1] == nkv and t.shape[3] == D and t.get_device() == q.get_device(),
              "attn_block: contiguous bfloat16 [., nkv, ., D] on one device")
    for t in (kv_len, row_len) + ((row_prompt,) if tables is None else ()) + ((row_cand,) if ck is not None else ()):
        _need(t is not None and t.dtype == torch.int32 and t.numel() == R and t.is_contiguous() and t.get_device() == q.get_device(), "attn_block: int32 [R] lengths and rows on q's device")
    _need(GT == G * T and k.shape == v.shape and (tables is None or (tables.dtype == torch.int32 and tables.dim() == 2 and tables.shape[0] == R and tables.stride(1) == 1 and tables.get_device() == q.get_device())) and
          (ck is None or (ck.shape == cv.shape and ck.shape[2] >= T)), "attn_block: shapes")
    out = torch.empty((R * T, nkv * G * D), dtype=q.dtype, device=q.device)
    max_keys = min(int(max_keys), k.shape[2] * (1 if tables is None else tables.shape[1]))
    splits, grouped = _block_plan(R * nkv, GT, max_keys, D)
    scratch = None
    if splits > 1:
        scratch = torch.empty((int(N.layers().jl_attn_block_scratch_floats(R, T, nkv, G, D, splits)),), dtype=torch.float32, device=q.device)
    a = N.BlockArgs(q=q.data_ptr(), k=k.data_ptr(), v=v.data_ptr(), ck=_ptr(ck), cv=_ptr(cv), kv_len=kv_len.data_ptr(), row_len=row_len.data_ptr(),
                    row_prompt=row_prompt.data_ptr() if tables is None else None, row_cand=row_cand.data_ptr() if ck is not None else None, tables=_ptr(tables), out=out.data_ptr(),
                    scratch=_ptr(scratch), table_ld=tables.stride(0) if tables is not None else 0, R=R, T=T, nkv=nkv, G=G, D=D, blocks=k.shape[0], page_size=k.shape[2],
                    table_cols=tables.shape[1] if tables is not None else 0, cand_rows=ck.shape[0] if ck is not None else 0, cand_max=ck.shape[2] if ck is not None else 0,
                    max_keys=max_keys, splits=splits, grouped=grouped, scale=D ** -0.5 if scale is None else float(scale))
    N.check_layers(N.layers().jl_attn_block(C.byref(a), _stream(q.device)), "jl_attn_block")
    return out


def attn_sweep_tile_rows(dtype: torch.dtype, H: int, G: int, D: int, Dv: int, k_cache: torch.Tensor, v_cache: torch.Tensor, value_heads: int = 0) -> int:
    """Queries per tile of the one-sweep kernel (heads in groups over a key head) for these sizes and pools; 0 when it does not
    take them."""
    if os.environ.get("JL_ATTN_NO_SWEEP") or (dtype == torch.float32 and (k_cache.data_ptr() % 16 or v_cache.data_ptr() % 16)):      # A/B switch for measurements; float rows are read 16 bytes at a time
        return 0
    v_in_k = v_cache.data_ptr() == k_cache.data_ptr()
    return int(N.layers().jl_attn_sweep_tile_rows(_code(dtype), H, G, value_heads or G, D, Dv, k_cache.stride(0), v_cache.stride(0), int(v_in_k)))


def attn_sweep(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, batch: RaggedBatch, H: int, G: int, D: int, Dv: int, scale: float,
               window: int, value_heads: int = 0, float_out: bool = False, sink: Optional[torch.Tensor] = None,
               gate: Optional[torch.Tensor] = None, gate_per_head: bool = False, chunk: int = 0, softcap: float = 0.0, out_scale: float = 1.0,
               out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Attention without bias or head mixing (``sink`` / ``gate`` / ``chunk`` / ``softcap`` / ``out_scale`` / ``out`` as for ``attn_window``) in one sweep on the matrix cores: q [N, H*D], pools as for
    ``attn_window`` (column ranges of wider rows allowed); ``v_cache`` may be the first Dv columns of ``k_cache`` itself (one key
    head whose rows hold the values: the latent pool).  Returns [N, H*Dv].  Sizes as ``attn_sweep_tile_rows`` accepts them."""
    _dev(q)
    n = q.shape[0]
    Gv = value_heads or G
    _need(q.is_contiguous() and q.shape[1] == H * D and n == batch.N and H % G == 0 and G % Gv == 0, "attn_sweep: q [N, H*D] of the batch")
    _need(k_cache.dtype == q.dtype and v_cache.dtype == q.dtype and k_cache.dim() == 2 and v_cache.dim() == 2 and k_cache.shape[1] == G * D and
          v_cache.shape[1] == Gv * Dv and k_cache.stride(1) == 1 and v_cache.stride(1) == 1 and k_cache.shape[0] == v_cache.shape[0],
          "attn_sweep: pool dtype / widths")
    _need(k_cache.shape[0] % batch.page_size == 0 and batch.max_page < k_cache.shape[0] // batch.page_size, "attn_sweep: a page lies outside the pool")
    _check_gate_sink(gate, sink, gate_per_head, n, H, Dv, q.dtype, "attn_sweep")
    tq = attn_sweep_tile_rows(q.dtype, H, G, D, Dv, k_cache, v_cache, Gv)
    _need(tq > 0, f"attn_sweep: heads={H} kv_heads={G} dim={D} vdim={Dv} are not sizes of this kernel")
    _need(chunk <= 0 or window <= 0, "attn_sweep: chunks exclude a window")
    out = _attn_out(out, n, H * Dv, torch.float32 if float_out else q.dtype, q.device, "attn_sweep")
    # few tiles with many keys (decoding): share each tile's keys out over workgroups until the chip is full
    tiles, groups = None, sum(-(-c // tq) for c in batch.counts) * G * -(-(H // G) // 32)
    # float tiles take 16 times as long per key, so the chip has to be fuller before their keys are left whole: 3 x 1000 tokens, 8 heads over 2 (648 groups)
    # 160 us shared out, 218 us in 128-row tiles; 1 x 4096 (1024 groups) 916 and 805 us
    below = SWEEP_SPLIT_BELOW_GROUPS if q.dtype == torch.bfloat16 else 2 * SWEEP_SPLIT_BELOW_GROUPS
    splits, scratch = 1, None
    if groups >= below and n >= SWEEP_WIDE_ROWS_PER_REQUEST * batch.B:
        # long portions: tiles of up to 128 (query, head) rows, every wavefront keeps its rows to itself
        wide = int(N.layers().jl_attn_sweep_wide_tile_rows(_code(q.dtype), H, G, Gv, D, Dv, k_cache.stride(0), v_cache.stride(0),
                                                           int(v_cache.data_ptr() == k_cache.data_ptr())))
        if wide > 0:
            # what starts last should be short (4 x 2048 tokens, 16 heads of 128 over 4 key heads: 175 -> 137 us).  The 32-row kernel keeps the
            # requests' order, in which neighbours share keys (over a latent of 512 the sorted order was 3 % slower)
            tq, tiles = wide, batch.tiles(wide, longest_first=True)
    narrow, few = False, 0
    if tiles is None and q.dtype == torch.bfloat16 and _fours(out) and not (q.data_ptr() | k_cache.data_ptr() | v_cache.data_ptr()) % 16 and \
            N.layers().jl_attn_narrow_ok(N.JL_BF16, H, G, Gv, D, Dv, k_cache.stride(0), v_cache.stride(0)):
        # few tokens per request: every wavefront with keys of its own
        narrow, tq = True, int(N.layers().jl_attn_talk_tile_rows(H, G, 0))
        tiles = batch.tiles(tq)
        reach = min(batch.max_pos, chunk + tq) if chunk > 0 else batch.max_pos if window <= 0 else min(batch.max_pos, int(window) + tq)
        few = _few(batch, H // G, 32, tq)
        splits = _token_splits(reach, tiles.shape[0] * G) if reach > NARROW_WHOLE else 1
        if splits > 1:
            scratch = torch.empty((int(N.layers().jl_attn_talk_scratch_floats(tiles.shape[0], tq, H, 1, Dv, splits)),), dtype=torch.float32, device=q.device)
    elif tiles is None:
        reach = min(batch.max_pos, chunk + tq) if chunk > 0 else batch.max_pos if window <= 0 else min(batch.max_pos, int(window) + tq)
        # the same over a latent: 32 rows up to 256 values, beyond 16, which read the keys twice as often (us, 4-wavefront tiles of 32 rows / so, latent of 512, 16 heads: 200 tokens at 1000 72 / 42, 1000 at none
        # 148 / 114, 2 x 1000 at 1000 321 / 324, 4 x 2000 998 / 1048)
        if v_cache.data_ptr() == k_cache.data_ptr() and q.dtype == torch.bfloat16 and _token_latent(H, D, Dv) and k_cache.stride(0) % 8 == 0 and _fours(out) and not (q.data_ptr() | k_cache.data_ptr()) % 16:
            few = _few(batch, H, 32, tq) if Dv <= 256 else _few(batch, H, 16, 16 // H) if H <= 16 and (groups < 2 * below or batch.N == batch.B) else 0
            # smaller tiles than the other form's may have to be copied where that one's came with the batch: not while a graph is captured
            if few and Dv > 256 and 16 // H not in batch._tiles and (batch._whole is None or batch._whole[0] > 16 // H) and torch.cuda.is_current_stream_capturing():
                few = 0
        if few:
            tq = tq if Dv <= 256 else 16 // H
            tiles = batch.tiles(tq)
            splits = _token_splits(reach, tiles.shape[0])
        elif groups < below:
            tiles = batch.tiles(tq)
            splits = max(1, min(-(-reach // 128), SWEEP_SPLIT_WORKGROUPS // groups, 64))
        if splits > 1:
            scratch = torch.empty((int(N.layers().jl_attn_sweep_scratch_floats(tiles.shape[0], H, G, Dv, splits)),), dtype=torch.float32, device=q.device)
    tiles = batch.tiles(tq) if tiles is None else tiles
    a = _attn_args(q, k_cache, v_cache, out, batch, tiles, gate, sink, None, None, None, scratch, None, scale, softcap, out_scale, H, G, Gv, D, Dv, window, 0, chunk, tq, splits,
                   N.JL_OUT_F32 if float_out else N.JL_OUT_SAME, gate_per_head)
    a.longest = few
    if narrow:
        N.check_layers(N.layers().jl_attn_narrow(C.byref(a), _stream(q.device)), "jl_attn_narrow")
        return out
    N.check_layers(N.layers().jl_attn_sweep(C.byref(a), _stream(q.device)), "jl_attn_sweep")
    return out


def retention_pieces_from(counts: Sequence[int], H: int, D: int) -> int:
    """From how many tokens on the requests of a step run in pieces, the others in the scan behind them (0: all in the scan).  Pieces of up to 32 tokens take 17 us at 128 x 128 and 30 for each
    256 heads of portions, the scan 6 and 0.75 per token of its longest portion, with more than 256 heads as much more; so all go to the scan where the longest portion is below a line that rises
    with the heads.  us, scan / pieces, 8 heads of 128: 8 tokens 12 / 17, 16 19 / 17, 8 x 16 19 / 23, 8 x 24 25 / 24, 16 x 24 26 / 32, 16 x 32 32 / 33, 32 x 32 37 / 45, 32 x 48 52 / 52, 64 x 48
    67 / 83, 128 x 64 159 / 157; 8 heads of 64: 16 14 / 13, 32 x 16 15 / 20, 32 x 32 25 / 21, 128 x 32 34 / 54, 128 x 64 68 / 74.  With single tokens beside, scan / pieces / both: 8 heads of 128,
    777 + 300 and 30 x 1 167 / 73 / 56, 8 x 16 and 32 x 1 24 / 53 / 34, 32 x 64 and 32 x 1 72 / 84 / 63; 16 heads of 64, 700, 40 x 10 and 40 x 1 121 / 78 / 69."""
    long = sum(c >= RETENTION_PIECES_FROM for c in counts)
    rounds = -(-long * H // 256)
    least = max(RETENTION_PIECES_FROM, min(4 * rounds, 16) if D > 64 else min(3 * rounds, 48), 3 + (len(counts) - long) * H // 230)
    if max(counts) < max(least, min(10 + long * H // 6, 64) if D > 64 else min(14 + long * H // 20, 72)):
        return 0
    return 1 if len(counts) * H < 256 else least                     # single tokens beside them where CUs are free: a launch less


def retention(proj: torch.Tensor, cols: Tuple[int, int, int, int], batch: RaggedBatch, H: int, D: int, Dv: int, rot_dims: int,
              cos: Optional[torch.Tensor], sin: Optional[torch.Tensor], decay: torch.Tensor, eps: float, state: torch.Tensor) -> torch.Tensor:
    """proj [N, ld] with q, k, v, gate at ``cols``; state [slots, H, D, Dv] float (updated in place).  Returns [N, H*Dv]."""
    _dev(proj)
    n, ld = proj.shape
    _need(proj.is_contiguous() and n == batch.N, "retention: proj [N, ld] of the batch")
    _need(state.dtype == torch.float32 and state.is_contiguous() and tuple(state.shape[1:]) == (H, D, Dv), "retention: state [slots, H, D, Dv] float")
    _need(batch.max_slot < state.shape[0], "retention: a slot lies outside the state")
    _need(decay.dtype == torch.float32 and decay.numel() == H, "retention: one decay per head")
    _need(max(cols[0], cols[1]) + H * D <= ld and max(cols[2], cols[3]) + H * Dv <= ld, "retention: columns do not fit the row")
    tl = 0
    if rot_dims:
        _need(cos is not None and cos.dtype == torch.float32 and cos.is_contiguous() and cos.shape == sin.shape and cos.shape[1] == rot_dims // 2,
              "retention: cos / sin [positions, rot_dims / 2] float")
        tl = cos.shape[0]
        _need(batch.max_pos <= tl, "retention: the angle tables are shorter than the batch's positions")
    out = torch.empty((n, H * Dv), dtype=proj.dtype, device=proj.device)
    L, st = N.layers(), _stream(proj.device)

    def scan(records, count, where, mode, what):
        N.check_layers(L.jl_retention(_ptr(proj), _code(proj.dtype), ld, cols[0], cols[1], cols[2], cols[3], _ptr(records), count, H, D, Dv,
                                      rot_dims, _ptr(cos), _ptr(sin), tl, _ptr(decay), float(eps), _ptr(where), _ptr(out), mode, st), what)

    least = batch._tiles.get(("retention", H, D))
    if least is None:
        least = batch._tiles[("retention", H, D)] = retention_pieces_from(batch.counts, H, D)
    if (least and L.jl_retention_pieces_ok(_code(proj.dtype), D, Dv, rot_dims) and ld % 4 == 0 and not any(c % 4 for c in cols[:3]) and
            proj.data_ptr() % (8 if proj.dtype == torch.bfloat16 else 16) == 0 and (not rot_dims or (cos.data_ptr() | sin.data_ptr()) % 16 == 0)):
        total = sum(c for c in batch.counts if c >= least)
        size = min(max(64, -(-total * H // RETENTION_WORKGROUPS) // 64 * 64), 1024)        # whole groups, as many pieces as the chip takes workgroups
        rec, req, rest = (*batch.pieces(size), None) if least == 1 else batch.long_pieces(size, least)[:3]
        scratch = torch.empty((rec.shape[0], H, D, Dv), dtype=torch.float32, device=proj.device)
        raw = torch.empty((n, H * Dv), dtype=torch.float32, device=proj.device)
        a = N.RetentionPieces(raw=raw.data_ptr(), N=n, proj=proj.data_ptr(), piece_rec=rec.data_ptr(), req=req.data_ptr(), pos=batch.pos.data_ptr(), cos_t=cos.data_ptr() if rot_dims else None,
                              sin_t=sin.data_ptr() if rot_dims else None, decay=decay.data_ptr(), state=state.data_ptr(), scratch=scratch.data_ptr(), out=out.data_ptr(), ld=ld,
                              table_len=tl, q_col=cols[0], k_col=cols[1], v_col=cols[2], g_col=cols[3], dtype=_code(proj.dtype), B=req.shape[0], pieces=rec.shape[0], piece_tokens=size,
                              H=H, D=D, Dv=Dv, rot_dims=rot_dims, eps=float(eps))
        N.check_layers(L.jl_retention_pieces_run(C.byref(a), st), "jl_retention_pieces_run")
        if rest is not None and rest.shape[0]:                       # behind it: its norm passes over all rows
            scan(rest, rest.shape[0], state, 0, "jl_retention")
        return out
    plan = batch.chunks(RETENTION_CHUNK)
    if plan is None:                                    # decoded tokens and short portions: one scan per request
        scan(batch.seq, batch.B, state, 0, "jl_retention")
        return out
    chunk_rec, chunk_len, req = plan
    scratch = torch.empty((chunk_rec.shape[0], H, D, Dv), dtype=torch.float32, device=proj.device)
    scan(chunk_rec, chunk_rec.shape[0], scratch, 1, "jl_retention(local state)")
    N.check_layers(L.jl_retention_join(_ptr(req), batch.B, _ptr(chunk_len), H, D, Dv, _ptr(decay), _ptr(state), _ptr(scratch), st), "jl_retention_join")
    scan(chunk_rec, chunk_rec.shape[0], scratch, 2, "jl_retention(outputs)")
    return out


ROUTER_OUTPUTS, ROUTER_TOKENS = 64, 32 * 512      # beyond: one launch for the choices and one workgroup for the grouping
ROUTER_DEPTH, ROUTER_DEPTH_FEW, ROUTER_FEW = 2048, 6144, 512      # router product in the same launch: depths times blocks of 16 outputs at most; for up to that many tokens (below)
_ROUTES = {"sigmoid": N.JL_ROUTE_SIGMOID, "softmax_renorm": N.JL_ROUTE_SOFTMAX_RENORM, "top_softmax": N.JL_ROUTE_TOP_SOFTMAX}


def _router_in_one(x: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor]) -> bool:
    """Whether the package's launches take the router product with the choice and the grouping: up to ROUTER_OUTPUTS outputs and ROUTER_TOKENS tokens, operands as ``linear`` takes them, and
    where that is not slower than ``linear`` in front of them.  Every 32 tokens take in all of W, so it is up to a product of the depth and the blocks of 16 outputs: ROUTER_DEPTH, for
    bfloat16 rows, which the library's product has to convert, 1.5 per token, and ROUTER_DEPTH_FEW for steps of up to ROUTER_FEW tokens, which wait for the host's launches.  us of GPU time with choice, grouping and small experts, product of its own / in one: 32 bfloat16 rows of 1024 by 16 outputs
    24 / 21, by 32 25 / 26, by 64 28 / 35; 1024 of 1024 by 32 33 / 31, of 2048 by 32 37 / 40, of 4096 by 64 48 / 86; 8192 of 1024 by 16 49 / 32, of 4096 by 64 100 / 101; float rows: 32 of 1024 by
    32 25 / 25, of 2048 by 32 25 / 32; 1024 of 1024 by 32 27 / 28, of 2048 by 32 29 / 37; 8192 of 2048 by 32 42 / 47.  us a pass of four layers, widths of 2048 by 32
    outputs: 32 decoding requests of Mikipel 817 / 796, of Lokizen 974 / 1012, one portion of 256 1106 / 1013, of 1000 1336 / 1352; by 40, 32 decoding requests of Voborax 1160 / 1119."""
    return (x.dim() == 2 and w.dim() == 2 and x.shape[1] * -(-w.shape[0] // 16) <= max(ROUTER_DEPTH_FEW if x.shape[0] <= ROUTER_FEW else ROUTER_DEPTH, 3 * x.shape[0] // 2 if x.dtype == torch.bfloat16 else 0) and _router_operands(x, w, bias))


def _router_operands(x: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor]) -> bool:
    return (x.dim() == 2 and 0 < x.shape[0] <= ROUTER_TOKENS and w.dim() == 2 and w.shape[0] <= ROUTER_OUTPUTS and x.dtype in _LINEAR_TYPES and w.dtype == torch.float32 and w.is_contiguous() and
            w.shape[1] == x.shape[1] and x.shape[1] % 4 == 0 and x.shape[1] > 0 and x.stride(1) == 1 and x.stride(0) >= x.shape[1] and x.stride(0) * x.element_size() % 16 == 0 and
            (x.data_ptr() | w.data_ptr()) % 16 == 0 and w.get_device() == x.get_device() and
            (bias is None or (bias.dtype == torch.float32 and bias.shape == (w.shape[0],) and bias.is_contiguous() and bias.get_device() == x.get_device())) and
            not (torch.is_grad_enabled() and (x.requires_grad or w.requires_grad or (bias is not None and bias.requires_grad))))


def moe_experts(h: torch.Tensor, router_logits: Optional[torch.Tensor], correction: Optional[torch.Tensor], top: int, scale: float,
                w_up: torch.Tensor, w_down: torch.Tensor, route: str = "sigmoid", renorm_eps: float = 0.0,
                gated: Optional[Tuple[int, float, float, float]] = None, identity: int = 0, router: Optional[Tuple[torch.Tensor, torch.Tensor, Optional[torch.Tensor]]] = None):
    """Routed experts: h [N, W], router_logits float [N, E] (or None and ``router`` = (x, w, bias) that they are ``linear``'s product of), w_down [E, W, ff].  Returns the weighted expert outputs per choice,
    float [N, top, W] (their sum over the middle axis is the layer's output).

    ``route`` "sigmoid": sigmoid scores, choice by score + correction, weights = score * scale; "softmax_renorm": softmax over all
    experts, the largest score + correction chosen, weights = score / (sum of the chosen scores + renorm_eps) * scale; "top_softmax": the largest logits chosen,
    weights = softmax over the chosen logits only, times scale.
    ``gated`` None: experts down(relu(up h)^2) with w_up [E, ff, W].  ``gated`` = (kind, limit, alpha, shift) of ``gated_act``: w_up
    [E, 2*ff, W] stacks every expert's gate rows on its linear rows, and the up product applies the unit in its epilogue.
    ``identity``: so many router outputs behind the E experts are identity experts, which have no weights and hand their input through.  Then
    returns (outputs, choice ids int32 [N, top], weights float [N, top]); the rows of outputs whose id is >= E are NOT written — what adds
    the outputs up (``output_norm``) puts weight * input in their place."""
    _dev(h)
    n, W = h.shape
    E, ff = w_down.shape[0], w_down.shape[2]
    Er = E + identity
    up_rows = 2 * ff if gated is not None else ff
    dev, dt = h.device, h.dtype
    in_one = router_logits is None and router is not None and _router_in_one(*router)
    if in_one:
        x, rw, rb = router
        _need(x.shape[0] == n and rw.shape[0] == Er and x.get_device() == h.get_device(), "moe_experts: router (x [N, K], w [experts + identity experts, K], bias) of h's rows")
    elif router_logits is None and router is not None:
        router_logits = linear(*router, float_out=True)
    _need(h.is_contiguous() and (in_one or (router_logits.dtype == torch.float32 and router_logits.is_contiguous() and tuple(router_logits.shape) == (n, Er))) and identity >= 0,
          "moe_experts: h [N, W], logits float [N, experts + identity experts]")
    _need(tuple(w_up.shape) == (E, up_rows, W) and tuple(w_down.shape) == (E, W, ff) and w_up.dtype == dt and w_down.dtype == dt and
          w_up.is_contiguous() and w_down.is_contiguous(), "moe_experts: expert weights [E, ff (2*ff when gated), W] / [E, W, ff] in the activation dtype")
    _need(route in _ROUTES and 1 <= top <= Er, "moe_experts: route is 'sigmoid', 'softmax_renorm' or 'top_softmax', 1 <= top <= experts")
    if correction is not None:
        _need(correction.dtype == torch.float32 and correction.numel() == Er, "moe_experts: correction float, one per router output")
    L, st = N.layers(), _stream(dev)
    rows = n * top
    tm = int(L.jl_moe_tile_rows(_code(dt), rows, E, W, ff))
    if tm == 128 and L.jl_moe_tile_pairs(rows, E, W, ff, int(gated is not None)):
        tm = 256
    elif tm == 64 and dt == torch.float32:
        tm = int(L.jl_moe_float_tiles(rows, E, W, ff))
    from_logits = not in_one and 0 < n <= ROUTER_TOKENS and Er <= ROUTER_OUTPUTS
    slices = int(L.jl_moe_router_slices(n, Er, router[0].shape[1])) if in_one else 1
    if (in_one or from_logits) and not os.environ.get("JL_MOE_UNFUSED_ACT"):
        r = (_H or _host()).moe_experts(h, *(router if in_one else (router_logits, None, None)), correction, top, scale, w_up, w_down, _ROUTES[route], renorm_eps, gated, identity, tm, slices)
        if r is not NotImplemented:
            return r
    ids = torch.empty((n, top), dtype=torch.int32, device=dev)
    wts = torch.empty((n, top), dtype=torch.float32, device=dev)
    # a decode's launches, which group nothing (moe_few_kernel and moe_router_few_kernel have the figures)
    if (in_one or from_logits) and tm == 32 and L.jl_moe_few_ok(_code(dt), n, Er, top, W, ff) and (h.data_ptr() | w_up.data_ptr() | w_down.data_ptr()) % 16 == 0 and not os.environ.get("JL_MOE_UNFUSED_ACT"):
        x, rw, rb = router if in_one else (router_logits, None, None)
        act, y = torch.empty((rows, ff), dtype=dt, device=dev), torch.empty((n, top, W), dtype=torch.float32, device=dev)
        a = N.MoeRouter(x=x.data_ptr(), w=_ptr(rw), bias=_ptr(rb), correction=_ptr(correction), ids=ids.data_ptr(), weights=wts.data_ptr(), N=n, x_ld=x.stride(0), x_dtype=_code(x.dtype),
                        K=x.shape[1], E=Er, experts=E, top=top, kind=_ROUTES[route], scale=float(scale), renorm_eps=float(renorm_eps))
        unit = gated or (0, 0.0, 0.0, 0.0)
        f = N.MoeFew(router=a, h=h.data_ptr(), w_up=w_up.data_ptr(), w_down=w_down.data_ptr(), act=act.data_ptr(), out=y.data_ptr(), dtype=_code(dt), W=W, ff=ff, gated=int(gated is not None),
                     unit=int(unit[0]), limit=float(unit[1]), alpha=float(unit[2]), shift=float(unit[3]))
        N.check_layers(L.jl_moe_few_run(C.byref(f), st), "jl_moe_few_run")
        return (y, ids, wts) if identity else y
    max_tiles = rows // tm + E
    blocks = int(L.jl_moe_router_blocks(n)) if in_one or from_logits else 0
    lists = torch.empty((rows + E + 2 + 2 * max_tiles + blocks * E + (slices * n * Er if slices > 1 else 0),), dtype=torch.int32, device=dev)       # the grouping's lists, one behind the other, the product's slices
    perm = lists.data_ptr()
    offsets = perm + 4 * rows
    tile_e = offsets + 4 * (E + 2)
    tile_r = tile_e + 4 * max_tiles
    if from_logits:
        x, rw, rb = router_logits, None, None
    if in_one or from_logits:
        a = N.MoeRouter(x=x.data_ptr(), w=_ptr(rw), bias=_ptr(rb), correction=_ptr(correction), ids=ids.data_ptr(), weights=wts.data_ptr(), perm=perm, offsets=offsets, tile_expert=tile_e,
                        tile_row0=tile_r, counts=tile_r + 4 * max_tiles, N=n, x_ld=x.stride(0), x_dtype=_code(x.dtype), K=x.shape[1], E=Er, experts=E, top=top, kind=_ROUTES[route],
                        tile_rows=tm, max_tiles=max_tiles, scale=float(scale), renorm_eps=float(renorm_eps), parts=tile_r + 4 * (max_tiles + blocks * E), slices=slices)
        N.check_layers(L.jl_moe_router_run(C.byref(a), st), "jl_moe_router_run")
    else:
        N.check_layers(L.jl_moe_route(_ptr(router_logits), _ptr(correction), n, Er, top, float(scale), _ptr(ids), _ptr(wts),
                                      _ROUTES[route], float(renorm_eps), st), "jl_moe_route")
        N.check_layers(L.jl_moe_group(_ptr(ids), n, top, E, tm, perm, offsets, tile_e, tile_r, max_tiles, st), "jl_moe_group")
    if gated is not None and not os.environ.get("JL_MOE_UNFUSED_ACT"):          # the unit in the product's epilogue (A/B switch for measurements)
        act = torch.empty((rows, ff), dtype=dt, device=dev)
        N.check_layers(L.jl_moe_gemm_gated(_ptr(h), _ptr(w_up), _code(dt), W, ff, top, perm, offsets, tile_e, tile_r, max_tiles, E, tm,
                                           int(gated[0]), float(gated[1]), float(gated[2]), float(gated[3]), _ptr(act), st), "jl_moe_gemm_gated")
    else:
        act = torch.empty((rows, up_rows), dtype=dt, device=dev)
        N.check_layers(L.jl_moe_gemm(_ptr(h), _ptr(w_up), _code(dt), N.JL_MOE_UP_PLAIN if gated is not None else N.JL_MOE_UP_RELU2, W, up_rows, top, perm,
                                     offsets, tile_e, tile_r, max_tiles, E, tm, None, _ptr(act), st), "jl_moe_gemm(up)")
        if gated is not None:
            act = gated_act(act, 0, ff, ff, *gated)
    y = torch.empty((n, top, W), dtype=torch.float32, device=dev)
    N.check_layers(L.jl_moe_gemm(_ptr(act), _ptr(w_down), _code(dt), N.JL_MOE_DOWN, ff, W, top, perm, offsets, tile_e, tile_r, max_tiles, E, tm,
                                 _ptr(wts), _ptr(y), st), "jl_moe_gemm(down)")
    return (y, ids, wts) if identity else y


ACT_GELU_TANH, ACT_CLAMPED_SWISH, ACT_SILU, ACT_GELU_ERF = N.JL_ACT_GELU_TANH, N.JL_ACT_CLAMPED_SWISH, N.JL_ACT_SILU, N.JL_ACT_GELU_ERF
ACT_SIGMOID, ACT_NONE = N.JL_ACT_SIGMOID, N.JL_ACT_NONE


def gated_act(z: torch.Tensor, g_col: int, u_col: int, F_: int, kind: int, limit: float = 0.0, alpha: float = 1.0, shift: float = 0.0,
              row_gate: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Gated activation of a feed-forward whose gate and linear branch are F_ columns each of one product z [N, ld], at g_col /
    u_col.  ACT_GELU_TANH: gelu_tanh(g) * u.  ACT_CLAMPED_SWISH: g' = min(g, limit), u' = clamp(u, +-limit), g' sigmoid(alpha g') (u' +
    shift).  ACT_SILU: g sigmoid(g) * u.  ACT_GELU_ERF: 0.5 g (1 + erf(g / sqrt 2)) * u.  ``u_col`` < 0: no linear branch (a plain
    activation of the F_ columns at g_col).  ``row_gate`` [N] or [N, 1] view (row stride free): the row is further multiplied by sigmoid(row_gate).  Returns [N, F_]."""
    _dev(z)
    r = (_H or _host()).gated_act(z, g_col, u_col, F_, kind, limit, alpha, shift, row_gate)
    if r is not NotImplemented:
        return r
    u_col = -1 if u_col < 0 else u_col
    _need(z.dim() == 2 and z.stride(1) == 1 and 0 <= g_col and g_col + F_ <= z.shape[1] and u_col + F_ <= z.shape[1], "gated_act: z [N, ld] with both column ranges inside")
    n = z.shape[0]
    rg_ld = 0
    if row_gate is not None:
        _need(row_gate.dtype == z.dtype and row_gate.numel() == n and row_gate.shape[0] == n, "gated_act: one row gate per row, of z's dtype")
        rg_ld = row_gate.stride(0)
    out = torch.empty((n, F_), dtype=z.dtype, device=z.device)
    N.check_layers(N.layers().jl_gated_act(_ptr(z), _code(z.dtype), n, z.stride(0), g_col, u_col, F_, int(kind), float(limit), float(alpha), float(shift),
                                          _ptr(row_gate), rg_ld, _ptr(out), _stream(z.device)), "jl_gated_act")
    return out


def scaled_add_norms(x: torch.Tensor, addends: Sequence[Tuple[torch.Tensor, Optional[torch.Tensor]]], w1: Optional[torch.Tensor],
                     w2: Optional[torch.Tensor], w_offset: float, eps: float, out_dtype: Optional[torch.dtype], two: bool = False,
                     second_float: bool = False):
    """x (float [N, W], in place) += sum over ``addends`` (y, scale) of scale * y, y [N, W] or [N, S, W] (summed over S) float or
    bfloat16, scale float [W] or None; then, with ``out_dtype``, the RMS norm of the updated x with float weights stored around
    ``w_offset``: x / rms(x) * (w_offset + w1) — and the same with w2 when ``two`` (both sublayers of a layer read one stream).
    Returns None, the norm, or the pair of norms; with ``second_float`` (and a 16-bit ``out_dtype``) a third tensor: the second norm
    unrounded, in float (for a float router beside the experts' 16-bit products)."""
    _dev(x)
    n, W = x.shape
    _need(x.dtype == torch.float32 and x.is_contiguous() and len(addends) <= 3, "scaled_add_norms: x contiguous float32 [N, W], at most 3 addends")
    arr = (N.Addend * max(1, len(addends)))()
    for k, (y, sc) in enumerate(addends):
        _need(y.is_contiguous() and y.shape[0] == n and y.shape[-1] == W and y.dim() in (2, 3), "scaled_add_norms: an addend is [N, W] or [N, S, W]")
        if sc is not None:
            _need(sc.dtype == torch.float32 and sc.numel() == W and sc.is_contiguous(), "scaled_add_norms: a scale is float [W]")
        arr[k] = N.Addend(y=y.data_ptr(), dtype=_code(y.dtype), count=1 if y.dim() == 2 else y.shape[1], scale=sc.data_ptr() if sc is not None else None)
    for w in (w1, w2):
        if w is not None:
            _need(w.dtype == torch.float32 and w.numel() == W and w.is_contiguous(), "scaled_add_norms: norm weights are float [W]")
    out1 = torch.empty((n, W), dtype=out_dtype, device=x.device) if out_dtype is not None else None
    out2 = torch.empty((n, W), dtype=out_dtype, device=x.device) if out_dtype is not None and two else None
    out2f = torch.empty((n, W), dtype=torch.float32, device=x.device) if out2 is not None and second_float and out_dtype != torch.float32 else None
    N.check_layers(N.layers().jl_scaled_add_norms(_ptr(x), arr, len(addends), _ptr(w1), _ptr(w2), float(w_offset), float(eps), _ptr(out1), _ptr(out2),
                                                 _ptr(out2f), _code(out_dtype or torch.float32), n, W, _stream(x.device)), "jl_scaled_add_norms")
    if two and second_float:
        return out1, out2, out2f if out2f is not None else out2
    return (out1, out2) if two else out1


def norm_add(x: torch.Tensor, y: torch.Tensor, g: torch.Tensor, eps: float, out_dtype: Optional[torch.dtype]) -> Optional[torch.Tensor]:
    """x (float [N, W], in place) += rms_norm(y) * g, g a single float (a norm on a sublayer's OUTPUT).  Returns x in
    ``out_dtype`` (None: the update only)."""
    _dev(x)
    n, W = x.shape
    _need(x.dtype == torch.float32 and x.is_contiguous() and y.is_contiguous() and tuple(y.shape) == (n, W), "norm_add: x float [N, W], y [N, W]")
    _need(g.dtype == torch.float32 and g.numel() == 1, "norm_add: the weight is one float")
    out = torch.empty((n, W), dtype=out_dtype, device=x.device) if out_dtype is not None else None
    N.check_layers(N.layers().jl_norm_add(_ptr(x), _ptr(y), _code(y.dtype), _ptr(g), float(eps), _ptr(out), _code(out_dtype or torch.float32), n, W,
                                         _stream(x.device)), "jl_norm_add")
    return out


NORM_RMS, NORM_LAYER = N.JL_NORM_RMS, N.JL_NORM_LAYER


def output_norm(x: torch.Tensor, addends: Sequence[Tuple[torch.Tensor, Optional[torch.Tensor]]], w: Optional[torch.Tensor], eps: float, kind: int, mult: float = 1.0,
                w_next: Optional[torch.Tensor] = None, out_dtype: Optional[torch.dtype] = None,
                choices: Optional[Tuple[torch.Tensor, torch.Tensor, int]] = None) -> Optional[torch.Tensor]:
    """x (float [N, W], in place) += mult * norm(sum of the addends) * w — a norm on a sublayer's OUTPUT, RMS (``NORM_RMS``) or layer norm
    (``NORM_LAYER``), w float [W]; addends (y [N, W] or [N, S, W], channel scale or None), at most three, none: no update.  Returns, in
    ``out_dtype`` (None: nothing), norm(x) * w_next, or x itself without ``w_next``.
    ``choices`` = (ids, weights, E): the first addend is what ``moe_experts`` returned with identity experts; choices >= E stand for
    weight * x (x before the update)."""
    _dev(x)
    r = (_H or _host()).output_norm(x, addends, w, eps, kind, mult, w_next, out_dtype, choices)
    if r is not NotImplemented:
        return r
    n, W = x.shape
    _need(x.dtype == torch.float32 and x.is_contiguous() and len(addends) <= 3, "output_norm: x contiguous float32 [N, W], at most 3 addends")
    arr = _addends(addends, n, W, "output_norm")
    for v in (w, w_next):
        _need(v is None or (v.dtype == torch.float32 and v.numel() == W and v.is_contiguous()), "output_norm: weights are float [W]")
    _need(w is not None or not addends, "output_norm: an update needs the norm's weight")
    ids = wts = None
    top = E = 0
    if choices is not None:
        ids, wts, E = choices
        _need(len(addends) >= 1 and addends[0][0].dim() == 3 and tuple(ids.shape) == tuple(wts.shape) == tuple(addends[0][0].shape[:2]) and ids.dtype == torch.int32 and
              wts.dtype == torch.float32 and ids.is_contiguous() and wts.is_contiguous(), "output_norm: choices int32 / float [N, top] of the first addend [N, top, W]")
        top = ids.shape[1]
    out = torch.empty((n, W), dtype=out_dtype, device=x.device) if out_dtype is not None else None
    N.check_layers(N.layers().jl_output_norm(_ptr(x), arr, len(addends), _ptr(ids), _ptr(wts), top, int(E), int(kind), _ptr(w), float(mult), float(eps), _ptr(w_next),
                                            _ptr(out), _code(out_dtype or torch.float32), n, W, _stream(x.device)), "jl_output_norm")
    return out


def product_f32(a: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """a [N, K] . w [M, K]^T with a float result [N, M] (not rounded to the operands' dtype): a product that becomes the residual stream."""
    return linear(a, w, float_out=True)


def sandwich_norm(x_in: torch.Tensor, y: Optional[torch.Tensor], w_post: Optional[torch.Tensor], eps: float, w_next: Optional[torch.Tensor] = None,
                  out_dtype: Optional[torch.dtype] = None, add_row: Optional[torch.Tensor] = None, out: Optional[torch.Tensor] = None,
                  plain: bool = False) -> Optional[torch.Tensor]:
    """x_in (float [N, W], in place) += rms_norm(y) * w_post + add_row (each part optional: y [N, W] with its norm weight, add_row float [W]);
    returns rms_norm(x_in) * w_next — or x_in itself with ``plain`` — in ``out_dtype`` or in ``out`` (a column range of wider rows); None with
    neither."""
    _dev(x_in)
    r = (_H or _host()).sandwich_norm(x_in, y, w_post, eps, w_next, out_dtype, add_row, out, plain)
    if r is not NotImplemented:
        return r
    n, W = x_in.shape
    _need(x_in.dtype == torch.float32 and x_in.is_contiguous(), "sandwich_norm: x contiguous float32 [N, W]")
    _need(y is None or (tuple(y.shape) == (n, W) and y.is_contiguous() and w_post is not None), "sandwich_norm: y [N, W] with its norm weight")
    for w in (w_post, add_row, w_next):
        _need(w is None or (w.dtype == torch.float32 and w.numel() == W and w.is_contiguous()), "sandwich_norm: weights and the added row are float [W]")
    if out is not None:
        _need(tuple(out.shape) == (n, W) and out.stride(1) == 1, "sandwich_norm: out [N, W], contiguous along a row")
    elif out_dtype is not None:
        out = torch.empty((n, W), dtype=out_dtype, device=x_in.device)
    _need(out is None or plain or w_next is not None, "sandwich_norm: the second norm needs its weight")
    N.check_layers(N.layers().jl_sandwich_norm(_ptr(x_in), _ptr(x_in), _ptr(y), _code(y.dtype) if y is not None else 0, _ptr(w_post), _ptr(add_row), float(eps),
                                              _ptr(w_next), _ptr(out), _code(out.dtype) if out is not None else 0, out.stride(0) if out is not None else 0,
                                              int(plain), n, W, _stream(x_in.device)), "jl_sandwich_norm")
    return out


def gated_norm(raw: torch.Tensor, gate: torch.Tensor, w: torch.Tensor, eps: float, act: int, gate_first: bool, parts: int = 1, scale: float = 1.0,
               out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """raw float [N, C] and its gate [N, C] (a column range of a product, row stride free): rms_norm over ``parts`` equal parts of the row of
    raw * act(gate) (``gate_first``), or of raw with act(gate) on the result; times w (float [C]) and ``scale``.  [N, C] of gate's dtype, in
    ``out`` (a column range of wider rows) when given."""
    _dev(raw)
    r = (_H or _host()).gated_norm(raw, gate, w, eps, act, gate_first, parts, scale, out)
    if r is not NotImplemented:
        return r
    n, C_ = raw.shape
    _need(raw.dtype == torch.float32 and raw.is_contiguous() and tuple(gate.shape) == (n, C_) and gate.stride(1) == 1, "gated_norm: raw float [N, C], gate [N, C]")
    _need(w.dtype == torch.float32 and w.numel() == C_ and w.is_contiguous() and parts >= 1 and C_ % parts == 0, "gated_norm: w float [C], parts that divide C")
    out = _attn_out(out, n, C_, gate.dtype, raw.device, "gated_norm")
    N.check_layers(N.layers().jl_gated_norm(_ptr(raw), _ptr(gate), _code(gate.dtype), gate.stride(0), _ptr(w), float(eps), int(act), int(gate_first), float(scale),
                                           _ptr(out), out.stride(0), n, C_, int(parts), _stream(raw.device)), "jl_gated_norm")
    return out


# A row alone (decoding for one user) and up to four go from a norm, a unit or a gate into the product in one launch, every workgroup of which makes the rows for itself (linear_after_kernel,
# jl_linear_after_ok); others take the two calls.  us a pass of one token through four layers, 1024 wide: 311 in launches of their own (49), 254 so (34).
def norm_linear(x: torch.Tensor, y: Optional[torch.Tensor], w_post: Optional[torch.Tensor], eps: float, w_next: torch.Tensor, add_row: Optional[torch.Tensor], w: torch.Tensor,
                bias: Optional[torch.Tensor] = None) -> Tuple[torch.Tensor, torch.Tensor]:
    """``sandwich_norm`` into w's dtype and ``linear`` of its result: the updated x (x itself, or another tensor, x as it was) and the product."""
    if not is_dynamo_compiling():
        r = (_H or _host()).norm_linear(x, y, w_post, eps, w_next, add_row, w, bias)
        if r is not NotImplemented:
            return r
    return x, linear(sandwich_norm(x, y, w_post, eps, w_next, w.dtype, add_row=add_row), w, bias)


def act_linear(z: torch.Tensor, g_col: int, u_col: int, F_: int, kind: int, w: torch.Tensor, bias: Optional[torch.Tensor] = None, limit: float = 0.0, alpha: float = 1.0, shift: float = 0.0) -> torch.Tensor:
    """``linear`` of ``gated_act``'s result."""
    if not is_dynamo_compiling():
        r = (_H or _host()).act_linear(z, g_col, u_col, F_, kind, limit, alpha, shift, w, bias)
        if r is not NotImplemented:
            return r
    return linear(gated_act(z, g_col, u_col, F_, kind, limit, alpha, shift), w, bias)


def feed_forward(x: torch.Tensor, w_gu: torch.Tensor, kind: int, w_down: torch.Tensor) -> torch.Tensor:
    """``linear`` by w_down of the gated unit (``gated_act``'s kinds without a limit) of ``linear`` by w_gu, whose rows are the gates and behind them the linear branches."""
    a = linear_gated(x, w_gu, kind)
    if a is not None:
        return linear(a, w_down)
    ff = w_down.shape[1]
    return act_linear(linear(x, w_gu), 0, ff, ff, kind, w_down)


def linear_gated(x: torch.Tensor, w_gu: torch.Tensor, kind: int, limit: float = 0.0, alpha: float = 1.0, shift: float = 0.0) -> Optional[torch.Tensor]:
    """``gated_act`` of ``linear``'s result, from the float sums, in the product's launch for some hundred to a few thousand rows (``linear_mid``); None where that does not take it.  us, 2048 rows of
    1024 by 2 x 2048: 24.9 and 5.9 for the unit, 24.5 so."""
    if is_dynamo_compiling():
        return None
    r = (_H or _host()).linear_gated(x, w_gu, kind, limit, alpha, shift)
    return None if r is NotImplemented else r


def gated_norm_linear(raw: torch.Tensor, gate: torch.Tensor, w_norm: torch.Tensor, eps: float, act: int, gate_first: bool, w: torch.Tensor, parts: int = 1, scale: float = 1.0) -> torch.Tensor:
    """``linear`` of ``gated_norm``'s result."""
    if parts == 1 and not is_dynamo_compiling():
        r = (_H or _host()).gated_norm_linear(raw, gate, w_norm, eps, act, gate_first, scale, w, None)
        if r is not NotImplemented:
            return r
    return linear(gated_norm(raw, gate, w_norm, eps, act, gate_first, parts, scale), w)


def polynorm(z: torch.Tensor, coef: torch.Tensor, eps: float) -> torch.Tensor:
    """c0 n(z) + c1 n(z^2) + c2 n(z^3) + c3 with n(u) = u / rms(u) over a row; z [N, F], coef four floats."""
    _dev(z)
    _need(z.dim() == 2 and z.is_contiguous() and coef.dtype == torch.float32 and coef.numel() == 4 and coef.is_contiguous(), "polynorm: z [N, F], coef float [4]")
    out = torch.empty_like(z)
    N.check_layers(N.layers().jl_polynorm(_ptr(z), _code(z.dtype), z.shape[0], z.shape[1], _ptr(coef), float(eps), _ptr(out), _stream(z.device)),
                   "jl_polynorm")
    return out


def causal_conv(x: torch.Tensor, w: torch.Tensor, batch: RaggedBatch, tail: Optional[torch.Tensor]) -> torch.Tensor:
    """x + (causal depthwise convolution of x over time, per request), from the float residual x [N, W] with w [W, taps]; ``tail``
    float [slots, taps - 1, W] carries every request's last inputs from step to step (updated here).  Returns [N, W] of w's dtype."""
    _dev(x)
    n, W = x.shape
    taps = w.shape[1]
    _need(x.dtype == torch.float32 and x.is_contiguous() and n == batch.N and w.is_contiguous() and w.shape[0] == W, "causal_conv: x float [N, W], w [W, taps]")
    if taps > 1:
        _need(tail is not None and tail.dtype == torch.float32 and tail.is_contiguous() and tuple(tail.shape[1:]) == (taps - 1, W) and
              batch.max_slot < tail.shape[0], "causal_conv: tail float [slots, taps - 1, W] with the batch's slots")
    out = torch.empty((n, W), dtype=w.dtype, device=x.device)
    L, st = N.layers(), _stream(x.device)
    N.check_layers(L.jl_causal_conv(_ptr(x), _ptr(w), _code(w.dtype), _ptr(batch.row_req), _ptr(batch.seq), _ptr(tail), n, W, taps, _ptr(out), st),
                   "jl_causal_conv")
    if taps > 1 and max(batch.counts) > 1:                  # single rows (decoding) have moved their tails in the launch above
        N.check_layers(L.jl_causal_conv_carry(_ptr(x), _ptr(batch.seq), batch.B, _ptr(tail), W, taps, st), "jl_causal_conv_carry")
    return out


def head_norm_append(proj: torch.Tensor, cols: Tuple[int, int, int], H: int, G: int, M: int, D: int, Dv: int, wq: Optional[torch.Tensor],
                     wk: Optional[torch.Tensor], eps: float, t_coef: float, t_every: int, batch: RaggedBatch, k_cache: torch.Tensor,
                     v_cache: torch.Tensor, maps_apart: bool = False, rot_dims: int = 0, cos: Optional[torch.Tensor] = None,
                     sin: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Per-head (and per score map) stage in front of attention: with ``rot_dims`` the rotation of q and k by position (rotate-half
    pairs on the first rot_dims dimensions of every head, angles from cos / sin [positions, rot_dims / 2] float), then the RMS norm
    of q and k over D (times wq / wk [D]; None: no weight), the query temperature by position, keys / values appended to the
    pools.  Returns q [N, M*H*D] map-major ([M, N, H*D] with ``maps_apart``: a contiguous query matrix per map); the key pool rows
    are [M, G, D] map-major."""
    _dev(proj)
    n, ld = proj.shape
    dt = proj.dtype
    _need(proj.is_contiguous() and n == batch.N, "head_norm_append: proj [N, ld] of the batch")
    for w in (wq, wk):
        _need(w is None or (w.numel() == D and w.dtype == dt), "head_norm_append: norm weights over one head")
    _need(rot_dims % 2 == 0 and 0 <= rot_dims <= D, "head_norm_append: the rotation takes an even number of dimensions up to D")
    _angle_tables(rot_dims, cos, sin, batch, "head_norm_append")
    _need(k_cache.dtype == dt and v_cache.dtype == dt and k_cache.is_contiguous() and v_cache.is_contiguous() and
          k_cache.shape[-1] == M * G * D and v_cache.shape[-1] == G * Dv and k_cache.shape[0] == v_cache.shape[0], "head_norm_append: pools [tokens, M*G*D] / [tokens, G*Dv]")
    q = torch.empty((M, n, H * D) if maps_apart else (n, M * H * D), dtype=dt, device=proj.device)
    N.check_layers(N.layers().jl_head_norm_append(_ptr(proj), _code(dt), n, ld, cols[0], cols[1], cols[2], H, G, M, D, Dv, _ptr(wq), _ptr(wk), float(eps),
                                                 float(t_coef), int(t_every), _ptr(batch.pos), _ptr(q), int(maps_apart), _ptr(k_cache), _ptr(v_cache),
                                                 _ptr(batch.kv_slot), int(rot_dims), _ptr(cos) if rot_dims else None, _ptr(sin) if rot_dims else None,
                                                 _stream(proj.device)), "jl_head_norm_append")
    return q


def diff_combine(a1: torch.Tensor, a2: torch.Tensor, H: int, Dv: int, lam: float, eps: float, out_scale: float, out_dtype: torch.dtype) -> torch.Tensor:
    """a1, a2 float [N, H*Dv] (two score maps' outputs; views with a common row stride) -> rms_norm_per_head(a1 - lam * a2) *
    out_scale, [N, H*Dv]."""
    _dev(a1)
    n = a1.shape[0]
    _need(a1.dtype == torch.float32 and a2.dtype == torch.float32 and tuple(a1.shape) == (n, H * Dv) and a2.shape == a1.shape and
          a1.stride(1) == 1 and a2.stride(1) == 1 and a1.stride(0) == a2.stride(0), "diff_combine: two float [N, H*Dv] with one row stride")
    out = torch.empty((n, H * Dv), dtype=out_dtype, device=a1.device)
    N.check_layers(N.layers().jl_diff_combine(_ptr(a1), _ptr(a2), a1.stride(0), n, H, Dv, float(lam), float(eps), float(out_scale), _ptr(out),
                                             _code(out_dtype), _stream(a1.device)), "jl_diff_combine")
    return out


def _angle_tables(rot_dims: int, cos, sin, batch: RaggedBatch, what: str) -> int:
    if not rot_dims:
        return 0
    _need(cos is not None and cos.dtype == torch.float32 and cos.is_contiguous() and cos.shape == sin.shape and cos.shape[1] == rot_dims // 2,
          f"{what}: cos / sin [positions, rot_dims / 2] float")
    _need(batch.max_pos <= cos.shape[0], f"{what}: the angle tables are shorter than the batch's positions")
    return cos.shape[0]


ROT_HALVES, ROT_NEIGHBOURS = N.JL_ROT_HALVES, N.JL_ROT_NEIGHBOURS      # which dimensions a rotation pairs: i with i + dims/2, or 2i with 2i + 1


def latent_prep(proj: torch.Tensor, q_col: int, Rq: int, kv_col: int, R: int, rd: int, rot_dims: int, wq: Optional[torch.Tensor], wkv: Optional[torch.Tensor],
                eps: float, batch: RaggedBatch, cos, sin, pool: Optional[torch.Tensor], pairing: int = N.JL_ROT_HALVES) -> Optional[torch.Tensor]:
    """Normalised query latent [N, Rq] (None with Rq = 0: a model without one); the pool row of every token becomes [normalised key/value
    latent | rotated shared key].  ``pool`` None: the query latent alone (a layer that attends over another layer's pool)."""
    _dev(proj)
    r = (_H or _host()).latent_prep(proj, q_col, Rq, kv_col, R, rd, rot_dims, wq, wkv, eps, batch.N, batch.max_pos, batch.pos, batch.kv_slot, cos, sin, pool, pairing)
    if r is not NotImplemented:
        return r
    n, ld = proj.shape
    dt = proj.dtype
    _need(proj.is_contiguous() and n == batch.N and (Rq == 0 or (wq is not None and wq.numel() == Rq and wq.dtype == dt)) and
          (pool is None or (wkv is not None and wkv.numel() == R and wkv.dtype == dt)),
          "latent_prep: proj [N, ld] of the batch, norm weights over the latents")
    _need(pool is None or (pool.dtype == dt and pool.is_contiguous() and pool.shape[-1] == R + rd), "latent_prep: pool [tokens, R + rd]")
    _need(pool is not None or Rq > 0, "latent_prep: neither a query latent nor a pool")
    if pool is None:
        R = rd = rot_dims = 0
    tl = _angle_tables(rot_dims, cos, sin, batch, "latent_prep")
    cq = torch.empty((n, Rq), dtype=dt, device=proj.device) if Rq else None
    N.check_layers(N.layers().jl_latent_prep(_ptr(proj), _code(dt), n, ld, q_col, Rq, kv_col, R, rd, rot_dims, _ptr(wq) if Rq else None, _ptr(wkv), float(eps),
                                            _ptr(batch.pos), _ptr(cos), _ptr(sin), tl, _ptr(cq), _ptr(pool), _ptr(batch.kv_slot), int(pairing),
                                            _stream(proj.device)), "jl_latent_prep")
    return cq


def latent_q_pack(qa: torch.Tensor, q: torch.Tensor, H: int, D: int, R: int, rd: int, rot_dims: int, batch: RaggedBatch, cos, sin,
                  pairing: int = N.JL_ROT_HALVES) -> torch.Tensor:
    """qa [H, N, R] (queries times the key up-projection), q [N, H*(D + rd)] (row stride free: a column range of a wider product) ->
    [N, H*(R + rd)] with the rotary part rotated."""
    _dev(q)
    r = (_H or _host()).latent_q_pack(qa, q, H, D, R, rd, rot_dims, batch.N, batch.max_pos, batch.pos, cos, sin, pairing)
    if r is not NotImplemented:
        return r
    n = q.shape[0]
    _need(q.stride(1) == 1 and qa.is_contiguous() and tuple(qa.shape) == (H, n, R) and q.shape[1] == H * (D + rd) and qa.dtype == q.dtype and n == batch.N,
          "latent_q_pack: qa [H, N, R], q [N, H*(D + rd)]")
    tl = _angle_tables(rot_dims, cos, sin, batch, "latent_q_pack")
    out = torch.empty((n, H * (R + rd)), dtype=q.dtype, device=q.device)
    N.check_layers(N.layers().jl_latent_q_pack(_ptr(qa), _ptr(q), q.stride(0), _code(q.dtype), n, H, D, R, rd, rot_dims, _ptr(batch.pos), _ptr(cos), _ptr(sin), tl,
                                              _ptr(out), int(pairing), _stream(q.device)), "jl_latent_q_pack")
    return out


def latent_attend(qf: torch.Tensor, pool: torch.Tensor, w_uv: torch.Tensor, batch: RaggedBatch, H: int, R: int, rd: int, scale: float, window: int,
                  sink: Optional[torch.Tensor] = None, gate: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Latent attention over the pool and the value up-projection behind it: qf [N, H*(R + rd)] (``latent_q_pack``), pool [tokens, R + rd]
    whose first R columns are the values, w_uv [H, R, Dv] -> [H, N, Dv].  ``window`` 0: plain causal; ``sink`` float [H]; ``gate`` [N, H] view:
    one sigmoid gate per head on its output (applied to the latent output: the up-projection is linear).  The launch is chosen by dtype and
    sizes; what no launch takes at once goes in column ranges of the latent, then in groups of heads."""
    n, W, dt = qf.shape[0], R + rd, qf.dtype
    per_head = gate is not None
    up = lambda o, c0, c1, h0, h1: (o.view(n, h1 - h0, c1 - c0).transpose(0, 1), w_uv[h0:h1] if c1 - c0 == R else w_uv[h0:h1, c0:c1].contiguous())
    if attn_sweep_tile_rows(dt, H, 1, W, R, pool, pool[:, :R]):                    # latents in multiples of 32 up to 512 (float: 128)
        o = attn_sweep(qf, pool, pool[:, :R], batch, H, 1, W, R, scale, window, sink=sink, gate=gate, gate_per_head=per_head)
        return torch.bmm(*up(o, 0, R, 0, H))
    fits = lambda h, c: int(N.layers().jl_attn_tile_rows(_code(dt), h, 1, W, c, pool.stride(0), pool.stride(0))) > 0
    heads, step = H, min(R, ATTN_MAX_VALUE_WIDTH) if dt == torch.bfloat16 else R   # bfloat16: the matrix-core kernel's value tile
    while not fits(heads, step) and (heads > 1 or step > 8):                       # columns in multiples of eight: the ranges stay aligned
        if step > 16 or heads == 1:
            step = (step // 2 + 7) // 8 * 8
        else:
            heads, step = -(-heads // 2), min(R, ATTN_MAX_VALUE_WIDTH)
    parts = []
    for h0 in range(0, H, heads):
        h1 = min(H, h0 + heads)
        q = qf if h1 - h0 == H else qf[:, h0 * W:h1 * W].contiguous()
        s_, g_ = sink[h0:h1].contiguous() if sink is not None else None, gate[:, h0:h1] if gate is not None else None
        ov = None
        for c0 in range(0, R, step):
            c1 = min(R, c0 + step)
            o = attn_window(q, g_, pool, pool[:, c0:c1], batch, h1 - h0, 1, W, c1 - c0, scale, window, 0, None, None, None, sink=s_, gate_per_head=per_head)
            o, wv = up(o, c0, c1, h0, h1)
            ov = torch.bmm(o, wv) if ov is None else torch.baddbmm(ov, o, wv)
        parts.append(ov)
    return parts[0] if len(parts) == 1 else torch.cat(parts, 0)


# What the two forms of latent attention run at (this card): attention over the latent on the 32-row tiles (wide; few: latents up to 256 in the launches for a few tokens) and (narrow latents, many rows) the 128-row tiles,
# attention over keys and values built per head, the product that builds them.  ``key`` is the time the built form takes per key of its longest tile when the
# chip is not full (a tile walks its keys in order; the 32-row kernel shares few tiles' keys out).  A layer wholly on built keys has fewer launches (bmm, packing, bmm
# and head order go: 95 -> 55 us of host time for small steps), a step that mixes the forms has more.  Not counted: the tables of the built form, 70 us of the host and 7 per request
# once per step, whatever the number of layers (8 prompts of 158 tokens, us a step over the latent / built: four layers 1357 / 1182, one layer 1168 / 1261).
LATENT_RATES = dict(narrow=330e12, few=240e12, wide=140e12, built=420e12, product=600e12, key64=25e-9, key32=50e-9, launches=-35e-6, both=80e-6)
# in float: the matrix form of the one-sweep kernel (narrow) or float multiply-adds (wide) over the latent
LATENT_RATES_FLOAT = dict(narrow=60e12, few=1.5e12, wide=1.5e12, built=60e12, product=90e12, key64=130e-9, key32=180e-9, launches=-35e-6, both=80e-6)
LATENT_BUILT_BYTES = 2 << 30          # keys and values built at a time
LATENT_BUILT_FROM = 16                # new tokens: no sizes make it worth building keys for fewer


def _latent_built_requests(batch: RaggedBatch, H: int, D: int, R: int, rd: int, Dv: int, window: int, dtype: torch.dtype = torch.bfloat16) -> List[int]:
    """The requests of a step whose keys and values are better built per head.  Over the latent a visible pair costs 2 H (2 R + rd) operations, over
    built keys 2 H (D + rd + Dv) — a third of it at R = 512, D = Dv = 128, rd = 64 — but every key is built first, 2 H R (D + Dv): worth it from some
    hundred new tokens per request on, never for a decoded token.  Measured, us over the latent / built: 4 x 1024 tokens at 16 heads x 128, R 512: 581 / 110,
    one request of 512 behind 4000: 430 / 300, of 128: 193 / 286, of 32: 108 / 258; 8 heads x 64, R 128, 4 x 256 behind 1500: 108 / 91, 1 x 256 behind 4000: 105 / 165."""
    key = ("built", H, D, R, rd, Dv, window, dtype)
    chosen = batch._tiles.get(key)
    if chosen is None:
        r = LATENT_RATES if dtype == torch.bfloat16 else LATENT_RATES_FLOAT
        over = 2.0 * H * (2 * R + rd) / (r["narrow"] if R <= 128 and R + rd <= 256 and batch.N * H >= 32 * SWEEP_SPLIT_BELOW_GROUPS else r["few"] if R <= 256 and _token_latent(H, R + rd, R) else r["wide"])
        pair, one = 2.0 * H * (D + rd + Dv) / r["built"], 2.0 * H * R * (D + Dv) / r["product"]
        step = r["key64"] if D + rd <= 128 else r["key32"]
        w, won, attend, chain, keys, chosen = window if window > 0 else 1 << 40, 0.0, 0.0, 0.0, 0, []
        for b, c in enumerate(batch.counts):
            if c < LATENT_BUILT_FROM:
                continue
            s = batch.starts[b]
            full = min(c, max(0, s + c - w))              # queries that see a whole window; the others see s + 1, s + 2, .. keys
            n, pairs = s + c - max(0, s - w + 1), full * w + (c - full) * (s + 0.5 * (1 + c - full))
            if (keys + n) * dtype.itemsize * H * (D + Dv) <= LATENT_BUILT_BYTES:
                chosen.append(b)
                won += pairs * over - n * one
                attend, chain, keys = attend + pairs * pair, max(chain, step * min(n, w + 127)), keys + n
        if won - max(attend, chain) <= (r["launches"] if len(chosen) == batch.B else r["both"]):
            chosen = []
        batch._tiles[key] = chosen
    return chosen


LATENT_HEADS = 8 << 20                # rows x heads x latent up to which the package forms the products of latent attention's heads


def latent_heads(n: int, H: int, D: int, R: int, Dv: int, dtype: torch.dtype) -> bool:
    """Whether the heads' products on both sides of attention over a latent are the package's launches, for n tokens.  us of GPU time, queries + outputs, library's products and their packing / own: 32
    tokens of 16 heads of 128, latent 512, 14.7 + 13.9 / 7.7 + 5.7, 1 token 13.1 + 14.4 / 4.1 + 5.0, 256 17.3 + 19.5 / 10.0 + 7.3, 512 22.1 + 15.4 / 15.5 + 14.8, 2000 of 8 heads, latent 256, 22.0 + 14.5 /
    15.6 + 10.3; at the line 1000 of 16 heads, latent 512, 34.3 + 18.6 / 30.4 + 22.2.  And 50 us less of the host."""
    return dtype == torch.bfloat16 and 0 < n * H * R <= LATENT_HEADS and D % 8 == 0 and R % 8 == 0 and Dv % 8 == 0


def latent_attention(q: torch.Tensor, pool: torch.Tensor, w_ukv: torch.Tensor, w_uk: torch.Tensor, w_uv: torch.Tensor, batch: RaggedBatch, H: int, D: int, R: int, rd: int, Dv: int, rot_dims: int,
                     cos, sin, pairing: int, scale: float, window: int, sink: Optional[torch.Tensor] = None, gate: Optional[torch.Tensor] = None,
                     gate_per_head: bool = False) -> torch.Tensor:
    """Latent attention from the queries to the heads' outputs [N, H*Dv]: q [N, H*(D + rd)] not yet rotated (row stride free; its rotary columns are
    OVERWRITTEN), pool [tokens, R + rd] with this step's rows in place, w_ukv [H*D + H*Dv, R] the key up-projections of all heads on the value up-projections,
    w_uk [H, D, R] and w_uv [H, R, Dv] the same per head, the latter turned.  ``window`` 0: plain causal; ``sink`` float [H]; ``gate`` a [N, H*Dv] view, or [N, H] with
    ``gate_per_head``: sigmoid gates on the outputs.
    Decoded tokens and short portions bring their queries to the latent (``latent_q_pack``, ``latent_attend``); for long portions in bfloat16 keys and values
    are built per head (``_latent_built_requests``) and attended on the 128-row tiles; a step may hold both.  Few tokens over the latent: the heads' products in launches of the package's own
    (``latent_heads``)."""
    _dev(q)
    n, dt = q.shape[0], q.dtype
    _need(q.dim() == 2 and q.stride(1) == 1 and q.shape[1] == H * (D + rd) and n == batch.N, "latent_attention: q [N, H*(D + rd)] of the batch")
    built: List[int] = []
    if D % 8 == 0 and rd % 8 == 0 and D + rd <= 256 and Dv % 32 == 0 and Dv <= 128 and q.stride(0) % 4 == 0 and q.data_ptr() % (2 * 4 if dt == torch.bfloat16 else 16) == 0 and R % 4 == 0:
        built = _latent_built_requests(batch, H, D, R, rd, Dv, window, dt)

    def over_latent(q, batch, gate):
        m = q.shape[0]
        if latent_heads(m, H, D, R, Dv, dt) and w_uk.shape == (H, D, R) and w_uv.shape == (H, R, Dv) and attn_sweep_tile_rows(dt, H, 1, R + rd, R, pool, pool[:, :R]):
            qf = (_H or _host()).latent_heads(q, w_uk, D + rd, rd, None, rot_dims, batch.N, batch.max_pos, batch.pos, cos, sin, pairing)
            if qf is not NotImplemented:
                o = attn_sweep(qf, pool, pool[:, :R], batch, H, 1, R + rd, R, scale, window, sink=sink, gate=gate if gate_per_head else None, gate_per_head=gate_per_head)
                r = (_H or _host()).latent_heads(o, w_uv, R, 0, None if gate_per_head else gate, 0, batch.N, batch.max_pos, batch.pos, None, None, pairing)
                if r is not NotImplemented:
                    return r
        qa = torch.bmm(q.view(m, H, D + rd)[:, :, :D].transpose(0, 1), w_uk)      # [H, N, R]: query . (W_uk c) = (W_uk^T query) . c
        qf = latent_q_pack(qa, q, H, D, R, rd, rot_dims, batch, cos, sin, pairing=pairing)
        return heads_gate(latent_attend(qf, pool, w_uv, batch, H, R, rd, scale, window, sink=sink, gate=gate if gate_per_head else None), None if gate_per_head else gate)

    if not built:
        return over_latent(q, batch, gate)
    _need(w_ukv.is_contiguous() and w_ukv.dtype == dt and tuple(w_ukv.shape) == (H * (D + Dv), R), "latent_attention: up-projections [H*D + H*Dv, R]")
    _need(pool.dtype == dt and pool.is_contiguous() and pool.shape[-1] == R + rd and pool.shape[0] % batch.page_size == 0 and
          batch.max_page < pool.shape[0] // batch.page_size, "latent_attention: pool [tokens, R + rd] that holds the batch's pages")
    _check_gate_sink(gate, sink, gate_per_head, n, H, Dv, dt, "latent_attention")
    out = torch.empty((n, H * Dv), dtype=dt, device=q.device)
    if len(built) < batch.B:                              # the other requests' rows, before the rotation below reaches them
        rest, rows = batch.part(sorted(set(range(batch.B)) - set(built)))
        out.index_copy_(0, rows, over_latent(q.index_select(0, rows), rest, None if gate is None else gate.index_select(0, rows)))
    keys, base = batch.key_rows(built, window)
    lat = pool.index_select(0, keys)
    kv = linear(lat[:, :R], w_ukv) if lat.dtype == torch.float32 else F.linear(lat[:, :R], w_ukv)
    tl = _angle_tables(rot_dims, cos, sin, batch, "latent_attention")
    st = _stream(q.device)
    N.check_layers(N.layers().jl_rotate_heads(_ptr(q), _code(dt), n, q.stride(0), H, D, rd, rot_dims, _ptr(batch.pos), _ptr(cos), _ptr(sin), tl, int(pairing), st), "jl_rotate_heads")
    tq, es = int(N.layers().jl_attn_expanded_tile_rows()), q.element_size()
    tiles = batch.tiles(tq, longest_first=True, requests=built)
    a = N.AttnArgs(q=q.data_ptr(), k_cache=kv.data_ptr(), v_cache=kv.data_ptr() + es * H * D, out=out.data_ptr(), tiles=tiles.data_ptr(), n_tiles=tiles.shape[0], H=H, G=H, D=D + rd,
                   Dv=Dv, window=int(window), TQ=tq, dtype=_code(dt), scale=float(scale), n_rows=n, k_ld=kv.shape[1], v_ld=kv.shape[1], Gv=H, out_dtype=N.JL_OUT_SAME,
                   sink=sink.data_ptr() if sink is not None else None, gate=gate.data_ptr() if gate is not None else None, gate_ld=gate.stride(0) if gate is not None else 0,
                   gate_heads=int(gate_per_head), out_scale=1.0, out_ld=H * Dv, key_base=base.data_ptr(), k_tail=lat.data_ptr() + es * R if rd else None, k_tail_ld=R + rd,
                   q_ld=q.stride(0), k_tail_cols=rd)
    N.check_layers(N.layers().jl_attn_expanded(C.byref(a), st), "jl_attn_expanded")
    return out


def heads_gate(ov: torch.Tensor, gate: Optional[torch.Tensor]) -> torch.Tensor:
    """ov [H, N, Dv] -> [N, H*Dv], times sigmoid(gate) (a [N, H*Dv] view, row stride free)."""
    _dev(ov)
    r = (_H or _host()).heads_gate(ov, gate)
    if r is not NotImplemented:
        return r
    H, n, Dv = ov.shape
    _need(ov.is_contiguous(), "heads_gate: ov [H, N, Dv] contiguous")
    if gate is not None:
        _need(gate.shape == (n, H * Dv) and gate.stride(1) == 1 and gate.dtype == ov.dtype, "heads_gate: gate [N, H*Dv]")
    out = torch.empty((n, H * Dv), dtype=ov.dtype, device=ov.device)
    N.check_layers(N.layers().jl_heads_gate(_ptr(ov), _ptr(gate), gate.stride(0) if gate is not None else 0, _code(ov.dtype), n, H, Dv, _ptr(out),
                                           _stream(ov.device)), "jl_heads_gate")
    return out


def _addends(addends, n: int, W: int, what: str):
    arr = (N.Addend * max(1, len(addends)))()
    for k, (y, sc) in enumerate(addends):
        _need(y.is_contiguous() and y.shape[0] == n and y.shape[-1] == W and y.dim() in (2, 3), f"{what}: an addend is [N, W] or [N, S, W]")
        if sc is not None:
            _need(sc.dtype == torch.float32 and sc.numel() == W and sc.is_contiguous(), f"{what}: a scale is float [W]")
        arr[k] = N.Addend(y=y.data_ptr(), dtype=_code(y.dtype), count=1 if y.dim() == 2 else y.shape[1], scale=sc.data_ptr() if sc is not None else None)
    return arr


def depth_mix_norm(x_in: torch.Tensor, addends: Sequence[Tuple[torch.Tensor, Optional[torch.Tensor]]], mult: float, streams: Optional[torch.Tensor],
                   depth: int, mix: Optional[torch.Tensor], x_out: Optional[torch.Tensor], w: Optional[torch.Tensor], eps: float,
                   out_dtype: Optional[torch.dtype], want_float: bool = False, shift: Optional[tuple] = None):
    """Residual update, weighted sum over the streams of all depths, RMS norm.  y = x_in + mult * sum of the addends ((tensor [N, W] or
    [N, S, W], channel scale or None), at most three).  With ``depth`` >= 0, y becomes streams[depth] (``streams`` float [depths, N, W]) and
    x_out = sum_{j <= depth} mix[j] * streams[j] (``mix`` float, at least depth + 1 entries; None: x_out = y); with ``depth`` < 0, x_out = y,
    or nothing is written when there are no addends.  Returns the norm of x_out (of x_in when nothing was written) times ``w`` (float
    [W] or None) in ``out_dtype`` — and, with ``want_float``, the same unrounded in float as a second result; None with neither.
    ``shift`` = (mu float [W], batch, tail float [slots, 1, W]): for a step in which every request brings ONE row, ``token_shift`` of the
    unrounded norm in the same launch; its result (``out_dtype``) is appended to what is returned."""
    _dev(x_in)
    if shift is None or (x_in.dim() == 2 and shift[1].N == shift[1].B == x_in.shape[0] and max(shift[1].counts) == 1):
        r = (_H or _host()).depth_mix_norm(x_in, addends, mult, streams, depth, mix, x_out, w, eps, out_dtype, want_float, None if shift is None else (shift[0], shift[2], shift[1].seq, shift[1].max_slot))
        if r is not NotImplemented:
            return r
    n, W = x_in.shape
    _need(x_in.dtype == torch.float32 and x_in.is_contiguous() and len(addends) <= 3, "depth_mix_norm: x_in contiguous float32 [N, W], at most 3 addends")
    arr = _addends(addends, n, W, "depth_mix_norm")
    written = depth >= 0 or len(addends) > 0
    if written:
        _need(x_out is not None and x_out.dtype == torch.float32 and x_out.is_contiguous() and x_out.shape == x_in.shape, "depth_mix_norm: x_out float [N, W]")
    ld = 0
    if depth >= 0:
        _need(streams is not None and streams.dtype == torch.float32 and streams.is_contiguous() and streams.dim() == 3 and tuple(streams.shape[1:]) == (n, W) and
              depth < streams.shape[0], "depth_mix_norm: streams float [depths, N, W] with room for this depth")
        ld = n * W
        if mix is not None:
            _need(mix.dtype == torch.float32 and mix.is_contiguous() and mix.numel() >= depth + 1, "depth_mix_norm: mix float with depth + 1 entries")
    if w is not None:
        _need(w.dtype == torch.float32 and w.numel() == W and w.is_contiguous(), "depth_mix_norm: the norm weight is float [W]")
    out = torch.empty((n, W), dtype=out_dtype, device=x_in.device) if out_dtype is not None else None
    outf = torch.empty((n, W), dtype=torch.float32, device=x_in.device) if want_float else None
    mu = seq = tail = outs = None
    if shift is not None:
        mu, batch, tail = shift
        _need(out_dtype is not None and batch.N == n and batch.B == n and max(batch.counts) == 1, "depth_mix_norm: the shift in this launch needs one row per request")
        _need(mu.dtype == torch.float32 and mu.numel() == W and mu.is_contiguous() and tail.dtype == torch.float32 and tail.is_contiguous() and
              tail.numel() == tail.shape[0] * W and batch.max_slot < tail.shape[0], "depth_mix_norm: mu float [W], tail float [slots, 1, W] with the batch's slots")
        seq, outs = batch.seq, torch.empty((n, W), dtype=out_dtype, device=x_in.device)
    N.check_layers(N.layers().jl_depth_mix_norm(_ptr(x_in), arr, len(addends), float(mult), _ptr(streams) if depth >= 0 else None, ld, int(depth),
                                               _ptr(mix) if depth >= 0 else None, _ptr(x_out) if written else None, _ptr(w), float(eps), _ptr(out),
                                               _code(out_dtype or torch.float32), _ptr(outf), n, W, _ptr(mu), _ptr(seq), _ptr(tail), _ptr(outs),
                                               _stream(x_in.device)), "jl_depth_mix_norm")
    res = (out, outf) if want_float else out
    if shift is not None:
        return (*res, outs) if want_float else (res, outs)
    return res


def token_shift(h: torch.Tensor, mu: torch.Tensor, batch: RaggedBatch, tail: torch.Tensor, out_dtype: torch.dtype) -> torch.Tensor:
    """h + (h of the previous token - h) * mu: h float [N, W], mu float [W]; ``tail`` float [slots, 1, W] carries every request's last h
    from step to step (updated here; never read by a request that starts at position 0)."""
    _dev(h)
    r = (_H or _host()).token_shift(h, mu, batch.N, batch.max_slot, batch.row_req, batch.seq, tail, out_dtype)
    if r is not NotImplemented:
        return r
    n, W = h.shape
    _need(h.dtype == torch.float32 and h.is_contiguous() and n == batch.N and mu.dtype == torch.float32 and mu.numel() == W and mu.is_contiguous(),
          "token_shift: h float [N, W] of the batch, mu float [W]")
    _need(tail.dtype == torch.float32 and tail.is_contiguous() and tail.numel() == tail.shape[0] * W and batch.max_slot < tail.shape[0],
          "token_shift: tail float [slots, 1, W] with the batch's slots")
    out = torch.empty((n, W), dtype=out_dtype, device=h.device)
    N.check_layers(N.layers().jl_token_shift(_ptr(h), _ptr(mu), _ptr(batch.row_req), _ptr(batch.seq), _ptr(tail), n, W, _ptr(out), _code(out_dtype),
                                            _stream(h.device)), "jl_token_shift")
    return out


def softcap(z: torch.Tensor, cap: float) -> torch.Tensor:
    """cap * tanh(z / cap), in place on contiguous float z."""
    _dev(z)
    _need(z.dtype == torch.float32 and z.is_contiguous() and cap > 0, "softcap: contiguous float32 values and a positive cap")
    N.check_layers(N.layers().jl_softcap(_ptr(z), z.numel(), float(cap), _stream(z.device)), "jl_softcap")
    return z


def softcap_float(z: torch.Tensor, cap: float) -> torch.Tensor:
    """cap * tanh(z / cap) as float: ``softcap`` of float z, and of bfloat16 z in the one pass that makes it float."""
    if z.dtype != torch.bfloat16:
        return softcap(z, cap)
    _dev(z)
    _need(z.is_contiguous() and cap > 0, "softcap_float: contiguous values and a positive cap")
    out = torch.empty(z.shape, dtype=torch.float32, device=z.device)
    N.check_layers(N.layers().jl_softcap_to(_ptr(z), _code(z.dtype), _ptr(out), z.numel(), float(cap), _stream(z.device)), "jl_softcap_to")
    return out


def short_conv(x: torch.Tensor, col: int, C_: int, w: torch.Tensor, batch: RaggedBatch, tail: Optional[torch.Tensor], act: int = N.JL_ACT_SILU,
               bias: Optional[torch.Tensor] = None, out_dtype: torch.dtype = torch.float32) -> torch.Tensor:
    """act(bias + causal depthwise convolution over time, per request) of the columns col .. col + C_ of x [N, ld], with w [C_, taps]; [N, C_]
    of ``out_dtype`` (float, or x's).  ``tail`` float [slots, taps - 1, C_] carries every request's last inputs from step to step (updated here)."""
    _dev(x)
    longest = batch._tiles.get("continued")
    if longest is None:                                  # the longest portion of a request that has a tail
        longest = batch._tiles["continued"] = max([c for c, s in zip(batch.counts, batch.starts) if s > 0], default=1)
    r = (_H or _host()).short_conv(x, col, C_, w, batch.N, batch.B, batch.max_slot, longest, batch.row_req, batch.seq, tail, act, bias, out_dtype)
    if r is not NotImplemented:
        return r
    n, ld = x.shape
    taps = w.shape[1]
    _need(x.is_contiguous() and n == batch.N and w.is_contiguous() and w.shape[0] == C_ and w.dtype == x.dtype and 0 <= col and col + C_ <= ld and 1 <= taps <= 8,
          "short_conv: x [N, ld] of the batch, w [C, taps <= 8] of its dtype, the columns inside the row")
    if taps > 1:
        _need(tail is not None and tail.dtype == torch.float32 and tail.is_contiguous() and tuple(tail.shape[1:]) == (taps - 1, C_) and
              batch.max_slot < tail.shape[0], "short_conv: tail float [slots, taps - 1, C] with the batch's slots")
    _need(bias is None or (bias.dtype == x.dtype and bias.numel() == C_ and bias.is_contiguous()), "short_conv: bias [C] of x's dtype")
    _need(out_dtype in (torch.float32, x.dtype), "short_conv: the output is float or of x's dtype")
    out = torch.empty((n, C_), dtype=out_dtype, device=x.device)
    N.check_layers(N.layers().jl_short_conv(_ptr(x), _code(x.dtype), ld, col, _ptr(w), _ptr(bias), _ptr(batch.row_req), _ptr(batch.seq), batch.B,
                                           longest, _ptr(tail), n, C_, taps, int(act), _ptr(out), _code(out_dtype), _stream(x.device)), "jl_short_conv")
    return out


def delta_chunks_from(counts: Sequence[int], H: int, D: int) -> int:
    """From how many tokens on the requests of a step go through the delta rule in chunks, the others behind them in the forms for short portions (0: none of them).  Portions of
    DELTA_CHUNKS_FROM tokens on are worth it alone; beside other requests the times of both ways are estimated, us per chunk of the longest, chunk and head, token of the columns' longest, token
    and head, request and head, token of the others' longest.  At widths of 64 the columns' walk is the faster one as soon as it fills the chip.  us, columns / chunks from 64 tokens on /
    this rule: 16 heads of 64, 100 x 100 233 / 288 / 231, 30 x 200 175 / 170 / 177; 8 heads of 128, 70 and 10 x 31 57 / 135 / 57, 300 + 63 178 / 93 / 51, 64 and 200 x 1 110 / 89 / 90,
    100 x 64 356 / 178 / 177.  (The times per chunk are those of a chain and chunks that took half as long again: the rule still finds the better way in these, by less.)"""
    if max(counts) < DELTA_CHUNKS_FROM or len(counts) == 1:
        return DELTA_CHUNKS_FROM if max(counts) >= DELTA_CHUNKS_FROM else 0
    first, chain, chunk, step, token, request, alone, single = (30, 6.7, 0.28, 0.6, 5.5e-3, 0.05, 2.7, 0.045) if D > 64 else (24, 4.9, 0.145, 0.49, 1.34e-3, 6e-3, 1.4, 0.012)
    c = sorted(counts)
    held = [0, *itertools.accumulate(c)]                  # tokens of the shortest ones

    def others(k):                                        # of the k shortest
        if k == 0:
            return 0.0
        longest, tokens, pairs = c[k - 1], held[k] * H, k * H
        if longest >= DELTA_COLUMNS_FROM:
            return 8 + max(step * longest, 0.6 * step * longest + token * tokens + request * pairs)
        return 8 + max(alone * longest, single * pairs + 0.012 * (tokens - pairs))

    best, least, k64 = others(len(c)), 0, bisect.bisect_left(c, 64)
    chunks = sum(-(-x // 64) for x in c[k64:])            # of 64 tokens and more; each shorter one is one
    for m in (2, 8, 16, DELTA_COLUMNS_FROM, 64):
        k = bisect.bisect_left(c, m)
        t = first + max(chain * -(-c[-1] // 64), chunk * H * (chunks + k64 - k)) + others(k)
        best, least = (t, m) if t < best else (best, least)
    return least


def delta_rule(qkv: torch.Tensor, cols: Tuple[int, int, int], proj: torch.Tensor, pcols: Tuple[int, int, int], a_log: torch.Tensor, dt_bias: torch.Tensor,
               norm_w: torch.Tensor, batch: RaggedBatch, H: int, G: int, D: int, Dv: int, unit_eps: float, q_scale: float, eps: float,
               state: torch.Tensor) -> torch.Tensor:
    """Gated delta rule.  qkv float [N, *] holds q, k (G*D each) and v (H*Dv) at ``cols`` (after convolution and activation); proj [N, ld]
    holds the decay input a, the step input b (H each) and the gate (H*Dv) at ``pcols``; a_log, dt_bias float [H]; norm_w float [Dv];
    state [slots, H, D, Dv] float (updated in place).  Returns [N, H*Dv] of proj's dtype."""
    _dev(proj)
    n, ld = proj.shape
    _need(proj.is_contiguous() and n == batch.N and qkv.dtype == torch.float32 and qkv.is_contiguous() and qkv.shape[0] == n, "delta_rule: proj and float qkv of the batch")
    _need(H % G == 0 and max(cols[0], cols[1]) + G * D <= qkv.shape[1] and cols[2] + H * Dv <= qkv.shape[1] and max(pcols[0], pcols[1]) + H <= ld and
          pcols[2] + H * Dv <= ld, "delta_rule: columns do not fit the rows")
    _need(state.dtype == torch.float32 and state.is_contiguous() and tuple(state.shape[1:]) == (H, D, Dv) and batch.max_slot < state.shape[0],
          "delta_rule: state float [slots, H, D, Dv] with the batch's slots")
    for t, k in ((a_log, H), (dt_bias, H), (norm_w, Dv)):
        _need(t.dtype == torch.float32 and t.is_contiguous() and t.numel() == k, "delta_rule: a_log, dt_bias float [H], norm_w float [Dv]")
    out = torch.empty((n, H * Dv), dtype=proj.dtype, device=proj.device)
    longest, least = max(batch.counts), batch._tiles.get(("delta", H, D))
    if least is None:
        least = batch._tiles[("delta", H, D)] = delta_chunks_from(batch.counts, H, D)
    if os.environ.get("JL_DELTA_NO_COLUMNS"):                               # A/B switch for measurements
        longest, least = 1, 0
    raw = torch.empty((n, H * Dv), dtype=torch.float32, device=proj.device) if longest >= DELTA_COLUMNS_FROM else None
    seq, B = batch.seq, batch.B
    if (least and N.layers().jl_delta_chunks_ok(D, Dv) and (qkv.shape[1] | cols[0] | cols[1]) % 4 == 0 and qkv.data_ptr() % 16 == 0):
        rec, req, seq, longest = batch.long_pieces(64, least)
        B, chunks, per = seq.shape[0], rec.shape[0], H // G
        floats = lambda heads: N.layers().jl_delta_chunks_floats(chunks, heads, H, G, D, Dv)
        heads = min(H, max(1, DELTA_SCRATCH_FLOATS // floats(per)) * per)
        scratch = torch.empty((floats(heads),), dtype=torch.float32, device=proj.device)
        columns = longest >= DELTA_COLUMNS_FROM                             # portions of lengths between: their launch norms and gates all rows
        a = N.DeltaChunks(qkv=qkv.data_ptr(), proj=proj.data_ptr(), A_log=a_log.data_ptr(), dt_bias=dt_bias.data_ptr(), norm_w=norm_w.data_ptr(), chunk_rec=rec.data_ptr(),
                          req=req.data_ptr(), state=state.data_ptr(), raw=raw.data_ptr(), scratch=scratch.data_ptr(), out=None if columns else out.data_ptr(), qkv_ld=qkv.shape[1],
                          ld=ld, N=n, scratch_floats=scratch.numel(), q_col=cols[0], k_col=cols[1], v_col=cols[2], a_col=pcols[0], b_col=pcols[1], g_col=pcols[2],
                          dtype=_code(proj.dtype), B=req.shape[0], chunks=chunks, H=H, G=G, D=D, Dv=Dv, pass_heads=heads, unit_eps=unit_eps, q_scale=q_scale, eps=eps)
        N.check_layers(N.layers().jl_delta_chunks_run(C.byref(a), _stream(proj.device)), "jl_delta_chunks_run")
        if B == 0:
            return out
        if not columns:
            raw = None                                                      # a workgroup per request and head, which writes its rows' outputs itself
    N.check_layers(N.layers().jl_delta_rule(_ptr(qkv), N.JL_F32, qkv.shape[1], cols[0], cols[1], cols[2], _ptr(proj), _code(proj.dtype), ld, pcols[0], pcols[1],
                                           pcols[2], _ptr(a_log), _ptr(dt_bias), _ptr(norm_w), _ptr(seq), B, n, H, G, D, Dv, float(unit_eps),
                                           float(q_scale), float(eps), _ptr(state), _ptr(raw), _ptr(out), _stream(proj.device)), "jl_delta_rule")
    return out


def scan_piece_groups(counts: Sequence[int], waves: int) -> int:
    """Groups of 64 tokens per piece of the linear recurrence, for ``waves`` wavefronts of 32 columns per request.  Portions that stay whole take one launch instead of three and half of the
    work, but walk their groups one after the other, 9 us each: up to two of them always, more where the requests' wavefronts fill the chip on average over that walk.  us, cut / whole, 64
    wavefronts per request: 40 tokens 21 / 16, 100 31 / 24, 192 32 / 32, 256 33 / 41, 3 x 192 40 / 34, 3 x 200 43 / 44, 8 x 200 62 / 47, 4 x 500 61 / 83, 8 x 500 109 / 88, 12 x 900 199 / 159,
    30 x 1000 419 / 282, 8 x 2000 283 / 334, 777 and 30 x 1 104 / 133; 8 per request: 30 x 300 38 / 39, 30 x 500 44 / 59.  Else as many pieces as fill the chip with two wavefronts per SIMD."""
    groups, longest = sum(-(-c // 64) for c in counts), -(-max(counts) // 64)
    if longest <= 2 or groups * waves >= 48 * longest * longest:
        return longest
    return max(1, min(8, sum(counts) * waves // (SCAN_WAVES * 64)))


def linear_scan(src: torch.Tensor, cols: Tuple[int, int, int], batch: RaggedBatch, H: int, G: int, D: int, Dv: int, state: torch.Tensor, act: int = N.JL_ACT_NONE,
                decay: Optional[torch.Tensor] = None, dt: Optional[torch.Tensor] = None, a_log: Optional[torch.Tensor] = None,
                dt_bias: Optional[torch.Tensor] = None, skip: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Linear recurrence S <- a S + k (u v)^T, o = S^T q + skip v per head.  src [N, ld] holds q, k (G*D each) and v (H*Dv) at ``cols``, which pass
    ``act`` on the way in.  ``decay`` float [H]: a = decay, u = 1; else u = softplus(dt + dt_bias), a = exp(-exp(a_log) u) with dt [N, H] (row
    stride free, src's dtype), a_log / dt_bias float [H].  skip float [H] or None.  state [slots, H, D, Dv] float, updated in place.  Returns
    float [N, H*Dv]."""
    _dev(src)
    if max(batch.counts) < SCAN_PIECES_FROM:
        r = (_H or _host()).linear_scan(src, *cols, batch.N, batch.B, batch.max_slot, batch.seq, H, G, D, Dv, state, act, decay, dt, a_log, dt_bias, skip)
        if r is not NotImplemented:
            return r
    n, ld = src.shape
    _need(src.stride(1) == 1 and n == batch.N and H % G == 0 and max(cols[0], cols[1]) + G * D <= ld and cols[2] + H * Dv <= ld, "linear_scan: columns of the batch's rows")
    _need(state.dtype == torch.float32 and state.is_contiguous() and tuple(state.shape[1:]) == (H, D, Dv) and batch.max_slot < state.shape[0],
          "linear_scan: state float [slots, H, D, Dv] with the batch's slots")
    _need(decay is not None or (dt is not None and a_log is not None and dt_bias is not None), "linear_scan: fixed decays, or dt with a_log and dt_bias")
    for t in (decay, a_log, dt_bias, skip):
        _need(t is None or (t.dtype == torch.float32 and t.is_contiguous() and t.numel() == H), "linear_scan: per-head constants are float [H]")
    if decay is None:
        _need(tuple(dt.shape) == (n, H) and dt.stride(1) == 1 and dt.dtype == src.dtype, "linear_scan: dt [N, H] of src's dtype")
    out = torch.empty((n, H * Dv), dtype=torch.float32, device=src.device)
    p = lambda t: t.data_ptr() if t is not None else None
    a = N.ScanArgs(src=p(src), dt=p(dt) if decay is None else None, decay=p(decay), A_log=p(a_log), dt_bias=p(dt_bias), skip=p(skip), seq=p(batch.seq), state=p(state), out=p(out),
                   ld=src.stride(0), dt_ld=dt.stride(0) if decay is None else 0, N=n, q_col=cols[0], k_col=cols[1], v_col=cols[2], dt_col=0, dtype=_code(src.dtype),
                   act=int(act), B=batch.B, H=H, G=G, D=D, Dv=Dv)
    if (max(batch.counts) >= SCAN_PIECES_FROM and not os.environ.get("JL_SCAN_NO_PIECES") and a.ld % 4 == 0 and all(c % 4 == 0 for c in cols) and    # A/B switch for measurements
            H * Dv <= 1 << 24 and Dv <= 1 << 22 and a.ld <= 1 << 26 and         # their kernel's offsets of 32 bits; the library sends wider calls to the scan by itself
            N.layers().jl_linear_scan_chunked_ok(a.dtype, D, Dv)):
        waves = H * -(-Dv // 32)
        size = batch._tiles.get(("scan", waves))
        if size is None:
            size = batch._tiles[("scan", waves)] = 64 * scan_piece_groups(batch.counts, waves)
        rec, req = batch.pieces(size)
        scratch = torch.empty((rec.shape[0] * H * (D * Dv + 1),), dtype=torch.float32, device=src.device)
        a.chunk_rec, a.req, a.scratch, a.chunks, a.B = p(rec), p(req), p(scratch), rec.shape[0], req.shape[0]
    N.check_layers(N.layers().jl_linear_scan(C.byref(a), _stream(src.device)), "jl_linear_scan")
    return out
