"""A decode's experts without a grouping (moe_router_few_kernel, moe_few_kernel over choices) at the edges of their tiles, against 64 bits."""
import pytest
import torch

from tests.test_moe_tiles import test_experts as check_experts

pytestmark = pytest.mark.gpu


# one token to the most, an expert's rows up to a tile, one and two more tiles and past them (all tokens choose the first), experts without rows, identity experts, choices beside 64 and 256 of them,
# depths below a stage, of whole stages and a rest, columns beside their 32
@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("N,E,top,W,ff,gated,identity,skew", [
    (1, 1, 1, 8, 8, False, 0, 0.0), (1, 16, 4, 1024, 512, False, 0, 0.0), (31, 3, 2, 72, 40, True, 0, 9.0), (32, 16, 4, 64, 136, False, 0, 30.0), (33, 5, 1, 136, 72, True, 2, 30.0),
    (64, 60, 4, 256, 96, True, 4, 0.0), (65, 4, 4, 96, 24, False, 0, 0.0), (96, 64, 8, 200, 64, False, 0, 30.0), (96, 6, 3, 320, 328, True, 1, 2.0), (17, 9, 5, 1000, 264, False, 0, 0.0),
])
def test_few_tokens(monkeypatch, dtype, N, E, top, W, ff, gated, identity, skew):
    from jacobiforcing_amd import _native as N_, layer_ops as LO
    lib, host, runs = N_.layers(), LO._host(), []
    assert lib.jl_moe_few_ok(LO._code(getattr(torch, dtype)), N, E + identity, top, W, ff)
    monkeypatch.setattr(lib, "jl_moe_tile_rows", lambda *a: 32, raising=False)
    check_experts(dtype, N, E, top, W, ff, gated, identity, skew)      # native

    class Without:
        def __getattr__(self, name):
            return (lambda *a: NotImplemented) if name == "moe_experts" else getattr(host, name)
    run = lib.jl_moe_few_run
    monkeypatch.setattr(LO, "_H", Without())
    monkeypatch.setattr(lib, "jl_moe_few_run", lambda *a: runs.append(1) or run(*a), raising=False)
    check_experts(dtype, N, E, top, W, ff, gated, identity, skew)      # the wrapper
    assert runs


def test_what_it_does_not_take():
    from jacobiforcing_amd import _native as N
    ok = N.layers().jl_moe_few_ok
    assert ok(N.JL_BF16, 96, 64, 8, 64, 64) and ok(N.JL_F32, 1, 1, 1, 4, 4)
    assert not any(ok(*a) for a in ((N.JL_BF16, 97, 8, 2, 64, 64), (N.JL_BF16, 96, 64, 11, 64, 64), (N.JL_BF16, 8, 65, 2, 64, 64), (N.JL_BF16, 8, 8, 2, 60, 64), (N.JL_F32, 8, 8, 2, 64, 62), (N.JL_BF16, 0, 8, 2, 64, 64)))
