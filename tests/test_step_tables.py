"""What a step's tables and rules on the host hold (no kernel runs)."""
import random

import numpy as np
import pytest
import torch

from jacobiforcing_amd import layer_ops as LO


def batch(counts, starts, page=64):
    need = [-(-(c + s) // page) for c, s in zip(counts, starts)]
    at = [sum(need[:b]) for b in range(len(need))]
    return LO.RaggedBatch.build(counts, starts, list(range(len(counts))), [list(range(a, a + n)) for a, n in zip(at, need)], page, "cpu")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_keys_built_per_head_stay_within_their_bytes(monkeypatch, dtype):
    """The bytes of keys and values that a step builds, in the activations' type."""
    H, D, R, rd, Dv = 16, 128, 512, 64, 128
    b = batch([4096] * 6, [0] * 6)
    per = 4096 * H * (D + Dv) * dtype.itemsize
    for room in (6, 3, 1):
        monkeypatch.setattr(LO, "LATENT_BUILT_BYTES", room * per)
        b._tiles.clear()
        chosen = LO._latent_built_requests(b, H, D, R, rd, Dv, 0, dtype)
        assert len(chosen) == room and sum(b.counts[i] for i in chosen) * H * (D + Dv) * dtype.itemsize <= LO.LATENT_BUILT_BYTES


@pytest.mark.parametrize("H,R,rd,token", [(32, 256, 64, True), (40, 256, 64, False), (8, 128, 64, True), (8, 128, 96, False), (16, 512, 64, False)])
def test_latents_are_priced_by_the_launch_that_takes_them(monkeypatch, H, R, rd, token):
    """A step over a latent counts at the rate of the launches for a few tokens where attention takes those (heads, rotary columns) and nowhere else."""
    assert LO._token_latent(H, R + rd, R) == (H <= 32 and R + rd <= R + 64)
    b, chosen = batch([1000], [0]), []
    for rate in (1e9, 1e18):
        monkeypatch.setitem(LO.LATENT_RATES, "few", rate)
        b._tiles.clear()
        chosen.append(LO._latent_built_requests(b, H, 128, R, rd, 128, 0))
    assert chosen == ([[0], []] if token else [chosen[0]] * 2)


def test_tiles_of_some_requests_keep_the_order_they_were_asked_for():
    b = batch([5, 3, 9], [0, 7, 2])
    for first in (False, True):
        b._tiles.clear()
        asked = [b.tiles(4, longest_first=x, requests=[1, 2]).tolist() for x in (first, not first)]
        in_order = asked[0] if not first else asked[1]
        assert in_order == [[1, 7, 3, 5], [2, 2, 4, 8], [2, 6, 4, 12], [2, 10, 1, 16]] and sorted(in_order, key=lambda r: -r[1]) == asked[1 if not first else 0]


def test_a_batch_without_its_tables_on_the_host():
    """One that was put together from its tensors: key rows and parts read them back."""
    import dataclasses
    b = batch([70, 3, 9], [0, 130, 2])
    bare = dataclasses.replace(b, _tiles={}, _host_tables=None)
    for window in (0, 50):
        assert all(torch.equal(x, y) for x, y in zip(b.key_rows([0, 1], window), bare.key_rows([0, 1], window)))
    (s1, r1), (s2, r2) = b.part([1, 2]), bare.part([1, 2])
    assert torch.equal(r1, r2) and torch.equal(s1.kv_slot, s2.kv_slot) and torch.equal(s1.tables, s2.tables)


@pytest.mark.parametrize("counts,starts,page,window", [([70, 3, 9], [0, 130, 2], 64, 0), ([70, 3, 9], [0, 130, 2], 64, 50), ([1, 33, 16, 65], [31, 0, 48, 640], 16, 17), ([5], [0], 1, 0),
                                                       ([64, 64], [64, 0], 64, 64), ([7, 2, 90], [100, 64, 3], 48, 1)])
def test_key_rows_are_those_of_the_pages_in_one_upload(monkeypatch, counts, starts, page, window):
    b = batch(counts, starts, page)
    for requests in (list(range(len(counts))), [len(counts) - 1], [0, len(counts) - 1][:len(counts)]):
        b._tiles.clear()
        want, base = [], [0] * len(counts)
        for r in requests:
            first = max(0, starts[r] - window + 1) if window else 0
            base[r] = len(want) - first
            want += [int(b.tables[r, p // page]) * page + p % page for p in range(first, starts[r] + counts[r])]
        uploads, to = [], torch.Tensor.to
        monkeypatch.setattr(torch.Tensor, "to", lambda t, *a, **k: uploads.append(t.shape) or to(t, *a, **k))
        tokens, places = b.key_rows(requests, window)
        monkeypatch.undo()
        assert tokens.dtype == torch.int64 and places.dtype == torch.int32 and tokens.tolist() == want and places.tolist() == base
        assert len(uploads) == 1                                        # each waits for everything queued before it


@pytest.mark.parametrize("seed", range(4))
def test_the_rule_is_the_cheapest_of_its_estimates(seed):
    """Against the same estimates over whole lists, for steps of all kinds; no kernel runs."""
    r = random.Random(seed)
    for _ in range(500):
        counts = [r.choice([1, r.randint(1, r.choice([3, 31, 64, 300, 2000]))]) for _ in range(r.randint(2, 60))] + [r.randint(64, 700)]
        H, D = r.choice([1, 4, 8, 16, 32]), r.choice([64, 128])
        c = np.asarray(counts)
        first, chain, chunk, step, token, request, alone, single = (30, 6.7, 0.28, 0.6, 5.5e-3, 0.05, 2.7, 0.045) if D > 64 else (24, 4.9, 0.145, 0.49, 1.34e-3, 6e-3, 1.4, 0.012)

        def others(r):
            if r.size == 0:
                return 0.0
            longest, tokens, pairs = int(r.max()), int(r.sum()) * H, r.size * H
            if longest >= LO.DELTA_COLUMNS_FROM:
                return 8 + max(step * longest, 0.6 * step * longest + token * tokens + request * pairs)
            return 8 + max(alone * longest, single * pairs + 0.012 * (tokens - pairs))

        ways = {0: others(c)}
        for m in (2, 8, 16, LO.DELTA_COLUMNS_FROM, 64):
            n = -(-c[c >= m] // 64)
            ways[m] = first + max(chain * int(n.max()), chunk * int(n.sum()) * H) + others(c[c < m])
        assert ways[LO.delta_chunks_from(counts, H, D)] == min(ways.values())


def test_requests_without_tokens_have_no_record_of_pieces():
    """The launches tell from more pieces than records that some request has several."""
    b = batch([0, 128, 0, 5], [7, 0, 0, 64])
    rec, req = b.pieces(64)
    assert rec.tolist() == [[0, 64, 1, 0], [64, 64, 1, 1], [128, 5, 3, 1]] and req.tolist() == [[0, 2, 0, 1], [2, 1, 64, 3]]


@pytest.mark.parametrize("counts", [[40, 7, 1], [31, 7], [100], [64, 65], [200, 1, 90]])
def test_pieces_that_come_with_the_tables(counts):
    """Portions that are one piece each have their records in the batch's own upload; the same as made on their own."""
    import dataclasses
    b = batch(counts, [3, 0, 70][:len(counts)])
    bare = dataclasses.replace(b, _tiles={}, _whole=None)
    for size in (64, 128, 256):
        got, want = b.pieces(size), bare.pieces(size)
        assert [t.tolist() for t in got] == [t.tolist() for t in want] and all(t.dtype == torch.int32 and t.is_contiguous() for t in got)
        assert (got[0].untyped_storage().data_ptr() == b.seq.untyped_storage().data_ptr()) == (32 <= max(counts) <= size)


def test_what_a_batch_is_built_of():
    """Page tables beyond the requests' are left out, but for the tables' width; lists of other lengths, positions that are not whole and counts below zero are refused."""
    build = lambda counts=[1, 70], starts=[2, 0], slots=[0, 1], tables=[[1], [2, 3], [4, 5, 6]]: LO.RaggedBatch.build(counts, starts, slots, tables, 64, "cpu")
    for counts in ([1, 70], [1, 1]):
        b = build(counts)
        assert b.tables.tolist() == [[1, -1, -1], [2, 3, -1]] and b.kv_slot[:2].tolist() == [66, 128] and b.max_page == 3
    whole = build(tables=torch.tensor([[1, 7], [2, 3], [4, 5]], dtype=torch.int32))
    assert whole.tables.tolist() == [[1, 7], [2, 3]] and whole.kv_slot[-1] == 3 * 64 + 5
    for bad in (dict(starts=[2, 0, 1]), dict(slots=[0, 1, 2]), dict(slots=[0]), dict(starts=[2.0, 0]), dict(counts=[1, -1]), dict(tables=[[1]])):
        with pytest.raises((ValueError, TypeError, IndexError)):
            build(**bad)


@pytest.mark.parametrize("counts,waves,groups", [([1, 40], 64, 1), ([128], 8, 2), ([129], 64, 1), ([200] * 3, 64, 4), ([200] * 3, 63, 1), ([500] * 4, 64, 1), ([500] * 8, 64, 8), ([2048] * 4, 64, 4), ([777] + [1] * 30, 64, 1),
                                                 ([1000] * 30, 64, 16), ([8192] * 8, 256, 8)])
def test_pieces_of_the_linear_recurrence(counts, waves, groups):
    """Whole up to two groups, or where the step's wavefronts fill the chip over the longest portion's walk; else as many as fill it, of at most eight groups."""
    assert LO.scan_piece_groups(counts, waves) == groups
