"""A step's tables formed in native code (jl_host.cpp) against the same formed in Python, over all forms that the native calls take; what they leave alone stays Python's to form or refuse."""
import random

import numpy as np
import pytest
import torch

from jacobiforcing_amd import layer_ops as LO

FIELDS = ("seq", "kv_slot", "tables", "row_req", "pos", "_host_tables")
NUMBERS = ("B", "N", "counts", "starts", "slots", "page_size", "max_pos", "max_page", "max_slot")


class _Counted:
    def __init__(self, real):
        self.real, self.taken = real, 0

    def __getattr__(self, name):
        def call(*a):
            r = getattr(self.real, name)(*a)
            self.taken += name in ("step_tables", "tile_records") and r is not NotImplemented
            return r
        return call


def _both(monkeypatch, *args):
    native = _Counted(LO._host())
    with monkeypatch.context() as m:
        m.setattr(LO, "_H", native)
        got = LO.RaggedBatch.build(*args, "cpu")
        m.setattr(LO, "_H", None)
        return got, LO.RaggedBatch.build(*args, "cpu"), native


def _same(a, b):
    for f in FIELDS:
        x, y = (np.asarray(getattr(t, f)) for t in (a, b))
        assert x.dtype == y.dtype and x.shape == y.shape and (x == y).all(), f
    assert all(getattr(a, f) == getattr(b, f) and type(getattr(a, f)) is type(getattr(b, f)) for f in NUMBERS)
    assert (a._whole is None) == (b._whole is None) and (a._whole is None or (a._whole[0], bool(a._whole[3])) == (b._whole[0], bool(b._whole[3])))


def test_tables_of_any_step(monkeypatch):
    rng = random.Random(5)
    for _ in range(300):
        B, page = rng.randint(1, 9), rng.choice([1, 3, 16, 48, 64])
        longest = rng.choice([1, 1, 2, LO.SCAN_PIECES_FROM, 200])
        counts, starts = [rng.randint(rng.choice([0, 1]), longest) for _ in range(B)], [rng.choice([0, rng.randint(0, 300)]) for _ in range(B)]
        tables = [[rng.randint(0, 10000) for _ in range(-(-(c + s) // page) + rng.choice([0, 0, 2]))] for c, s in zip(counts, starts)]
        tables += [[7] * rng.randint(0, 30)] * rng.choice([0, 0, 1])
        as_kind = rng.choice([list, tuple])
        a, b, native = _both(monkeypatch, as_kind(counts), as_kind(starts), as_kind(rng.randint(0, 99) for _ in range(B)), as_kind(map(rng.choice([list, tuple]), tables)), page)
        assert native.taken == 1
        _same(a, b)
        for tq in (1, 4, 7, 32, longest):
            for first in (False, True):
                with monkeypatch.context() as m:
                    m.setattr(LO, "_H", native)
                    x = a.tiles(tq, longest_first=first)
                assert x.dtype == torch.int32 and torch.equal(x, b.tiles(tq, longest_first=first))
        if a._whole is not None and a._whole[3]:
            assert all(torch.equal(x, y) for x, y in zip(a.pieces(256), b.pieces(256)))


@pytest.mark.parametrize("args", [
    ([1, 2], [0, 5], [0, 1], [np.asarray([3]), np.asarray([4])], 64), (np.asarray([3]), [0], [0], [[1]], 64), ([1], [0], [0], [[1 << 40]], 64), ([True], [0], [0], [[1]], 64), ([2.0], [0], [0], [[1]], 64),
    ([1], [5], [1 << 33], [[1]], 64),
])
def test_other_kinds_of_numbers_are_formed_as_before(monkeypatch, args):
    def tried(native):
        with monkeypatch.context() as m:
            m.setattr(LO, "_H", native)
            try:
                return LO.RaggedBatch.build(*args, "cpu")
            except Exception as e:
                return type(e), str(e)
    native = _Counted(LO._host())
    a, b = tried(native), tried(None)
    assert native.taken == 0
    if isinstance(b, tuple):
        assert a == b
    else:
        _same(a, b)


@pytest.mark.parametrize("args", [
    ([1, 2], [0], [0, 1], [[1], [2]], 64), ([65], [0], [0], [[1]], 64), ([-1], [0], [0], [[1]], 64), ([], [], [], [], 64), ([1], [0], [0], [], 64), ([1], [0], [0], [[1]], 0), ([1], ["0"], [0], [[1]], 64),
    ([1, 1], [0, 64], [0, 1], [[1], [2]], 64), (None, [0], [0], [[1]], 64),
])
def test_what_is_refused_stays_refused(monkeypatch, args):
    seen = []
    for native in (_Counted(LO._host()), None):
        with monkeypatch.context() as m:
            m.setattr(LO, "_H", native)
            with pytest.raises(Exception) as e:
                LO.RaggedBatch.build(*args, "cpu")
        seen.append((type(e.value), str(e.value)))
        assert native is None or native.taken == 0
    assert seen[0] == seen[1]
