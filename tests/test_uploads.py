"""A step's tables: what they hold, request by request, and that they reach the device without waiting for queued kernels, whole for every stream, and keep their memory until kernels are done with it."""
import random

import numpy as np
import pytest
import torch

from jacobiforcing_amd import layer_ops as LO


def tables(counts, starts, slots, pages, size):
    """Token by token."""
    seq, kv, req, pos, r0 = [], [], [], [], 0
    for b, (c, s) in enumerate(zip(counts, starts)):
        seq.append([r0, c, s, slots[b]])
        kv += [int(pages[b][p // size]) * size + p % size for p in range(s, s + c)]
        req += [b] * c
        pos += range(s, s + c)
        r0 += c
    return seq, kv, req, pos


@pytest.mark.parametrize("seed", range(12))
def test_tables_on_the_host(seed):
    """Portions, single tokens and requests without any; tables of one length and of several, lists and arrays; spare pages; tiles that come with the tables and tiles that do not."""
    rng = random.Random(seed)
    B, size = rng.randint(1, 9), rng.choice([1, 7, 64])
    counts = [1] * B if seed % 3 == 0 else [rng.choice([0, 1, rng.randint(2, 90)]) if seed % 3 == 1 else rng.randint(1, 40) for _ in range(B)]
    starts, slots = [rng.randint(0, 200) for _ in range(B)], rng.sample(range(50), B)
    pages = [[rng.randint(0, 999) for _ in range(-(-(c + s) // size) + rng.choice([0, 0, 2]))] for c, s in zip(counts, starts)]
    given = [np.asarray(p, dtype=np.int32) if rng.random() < 0.3 else p for p in pages]
    b = LO.RaggedBatch.build(counts, starts, slots, given, size, "cpu")
    seq, kv, req, pos = tables(counts, starts, slots, pages, size)
    assert (b.seq.tolist(), b.kv_slot.tolist(), b.row_req.tolist(), b.pos.tolist()) == (seq, kv, req, pos)
    assert [[x for x in row if x >= 0] for row in b.tables.tolist()] == pages and b.tables.shape == (B, max(1, max(map(len, pages))))
    assert (b.N, b.max_pos, b.max_slot, b.max_page) == (sum(counts), max(s + c for s, c in zip(starts, counts)), max(slots), max(max(p, default=-1) for p in pages))
    for tq in (1, 8, 100):
        want = [[i, s + o, min(tq, c - o), r[0] + o] for i, (c, s, r) in enumerate(zip(counts, starts, seq)) for o in range(0, c, tq)]
        assert b.tiles(tq).tolist() == want and b.tiles(tq).dtype == torch.int32
    with pytest.raises(ValueError, match="do not hold"):
        LO.RaggedBatch.build([5], [3 * size], [0], [[0, 1, 2]], size, "cpu")


@pytest.mark.gpu
def test_tables_do_not_wait_and_last():
    """Behind a long queue: tables are whole for another stream at once, and those of many steps, each dropped as soon as its kernel is queued, are what the kernels read in the end."""
    x = torch.randn(8192, 8192, device="cuda").bfloat16()
    x @ x
    torch.cuda.synchronize()
    queued = torch.cuda.Event()
    for _ in range(300):                                     # hundreds of milliseconds
        y = x @ x
    queued.record()
    first = LO.RaggedBatch.build([40], [0], [0], [list(range(8))], 64, "cuda")
    assert not queued.query(), "the tables waited for the queue"
    got = torch.empty(200, 40, dtype=torch.int64, device="cuda")
    other = torch.cuda.Stream()
    for i in range(200):
        b = LO.RaggedBatch.build([40], [i], [0], [list(range(i, i + 8))], 64, "cuda") if i else first
        if i % 50 == 0:
            with torch.cuda.stream(other):
                seen = b.kv_slot.clone()
            other.synchronize()
            assert seen.tolist() == tables([40], [i], [0], [list(range(i, i + 8))], 64)[1]
        got[i].copy_(b.kv_slot)
        del b
    torch.cuda.synchronize()
    assert got.tolist() == [tables([40], [i], [0], [list(range(i, i + 8))], 64)[1] for i in range(200)] and bool(y.isfinite().all())


@pytest.mark.gpu
def test_tables_that_another_stream_reads(monkeypatch):
    """A batch built on one stream, read behind a queue on another and dropped: its memory is not written before the first stream, which waits for the other, is through."""
    monkeypatch.setattr(LO, "GONE_AT_ONCE", 1)
    x, other, here = torch.randn(8192, 8192, device="cuda").bfloat16(), torch.cuda.Stream(), torch.cuda.current_stream()
    for start in (7, 3):
        b = LO.RaggedBatch.build([40], [start], [0], [[5, 9, 2]], 64, "cuda")
        torch.cuda.synchronize()
        with torch.cuda.stream(other):
            for _ in range(20):
                y = x @ x
            seen = torch.stack([b.kv_slot, b.kv_slot])[1]
        del b
        here.wait_stream(other)
        more = [LO.RaggedBatch.build([40], [i], [0], [list(range(i, i + 8))], 64, "cuda") for i in range(20)]
        torch.cuda.synchronize()
        assert seen.tolist() == tables([40], [start], [0], [[5, 9, 2]], 64)[1] and bool(y.isfinite().all())
        assert all(m.kv_slot.tolist() == tables([40], [i], [0], [list(range(i, i + 8))], 64)[1] for i, m in enumerate(more))


@pytest.mark.gpu
@pytest.mark.filterwarnings("ignore:The CUDA Graph is empty")
def test_tables_are_refused_in_a_capture():
    """... before anything that would leave an error behind."""
    build = lambda: LO.RaggedBatch.build([3, 1], [0, 5], [0, 1], [[0], [1]], 64, "cuda")
    b = build()
    with pytest.raises(RuntimeError, match="captured"), torch.cuda.graph(torch.cuda.CUDAGraph()):
        build()
    with pytest.raises(RuntimeError, match="captured"), torch.cuda.graph(torch.cuda.CUDAGraph()):
        b.pieces(64)
    torch.cuda.synchronize()
    assert build().pos.tolist() == [0, 1, 2, 5] and b.pieces(64)[1].tolist() == [[0, 1, 0, 0], [1, 1, 5, 1]]


@pytest.mark.gpu
def test_what_is_kept_is_given_back(monkeypatch):
    """Tables of batches that are gone wait for one event at a time and then go, but for those that somebody kept a part of, which stay whole."""
    monkeypatch.setattr(LO, "GONE_AT_ONCE", 8)
    build = lambda i: LO.RaggedBatch.build([40], [i], [0], [list(range(i, i + 8))], 64, "cuda")
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        kept = [build(i).kv_slot[3:] for i in range(20)]
        for i in range(300):
            b = build(i % 100)
            b.pieces(64)
        torch.cuda.synchronize()
        gone = next(g for g in LO._GONE.values() if g.stream == stream)
        for i in range(2 * LO.GONE_AT_ONCE):                     # two sweeps more: the first finds all events passed
            b = build(i)
        assert len(gone.tables) <= LO.GONE_AT_ONCE and sum(len(left) for _, left in gone.waiting) <= 3 * LO.GONE_AT_ONCE
        torch.cuda.synchronize()
        assert all(t.tolist() == tables([40], [i], [0], [list(range(i, i + 8))], 64)[1][3:] for i, t in enumerate(kept))
