"""Routed experts in tiles of 256 rows: the way up by one workgroup per CU, the way down in halves of the tiles, at the edges of tiles, columns, depths and rounds, against 64 bits."""
import pytest
import torch

from tests.test_moe_tiles import test_experts as check_experts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,E,top,W,ff,gated,identity,skew", [
    (1, 2, 1, 64, 64, True, 0, 0.0), (128, 1, 1, 64, 128, True, 0, 0.0), (129, 1, 1, 128, 136, True, 0, 0.0), (256, 1, 1, 192, 256, False, 0, 0.0), (257, 1, 1, 64, 264, False, 0, 0.0),
    (700, 3, 2, 320, 96, True, 1, 2.0), (513, 9, 1, 1024, 520, True, 0, 9.0), (640, 40, 2, 64, 512, False, 4, 3.0), (300, 5, 2, 72, 40, True, 0, 0.0), (300, 5, 2, 64, 50, True, 0, 0.0),
    (3000, 8, 4, 128, 1160, True, 0, 1.0), (9000, 3, 3, 64, 2056, False, 0, 0.0),
])
def test_tiles_of_256_rows(monkeypatch, N, E, top, W, ff, gated, identity, skew):
    """One tile, several per workgroup (the last two: 500 tiles for 256 workgroups and more), incomplete ones of at most 128 rows and of more; depths that the kernel for 256 rows does not take."""
    from jacobiforcing_amd import _native as N_
    asked = []
    monkeypatch.setattr(N_.layers(), "jl_moe_tile_rows", lambda *a: asked.append(a) or 256, raising=False)
    check_experts("bfloat16", N, E, top, W, ff, gated, identity, skew)
    assert asked


@pytest.mark.parametrize("gated", [True, False])
def test_pairs_that_the_rule_chooses(gated):
    from jacobiforcing_amd import _native as N_
    lib = N_.layers()
    N, E, top, W, ff = 8192, 12, 4, 256, 1024 if gated else 1280
    assert lib.jl_moe_tile_rows(N_.JL_BF16, N * top, E, W, ff) == 128 and lib.jl_moe_tile_pairs(N * top, E, W, ff, int(gated)) == 1
    assert not lib.jl_moe_tile_pairs(N * top, E, W + 8, ff, int(gated)) and not lib.jl_moe_tile_pairs(255 * E, E, W, 1 << 20, int(gated))
    check_experts("bfloat16", N, E, top, W, ff, gated, 0, 0.0)
