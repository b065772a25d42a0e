"""What a step's tables and rules on the host hold (no kernel runs)."""
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
