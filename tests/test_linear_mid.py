"""Dense products of some hundred to a few thousand rows (linear_mid_kernel) at the edges of its tiles, depths and results, against the same in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _operands(n, k, o, ld, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(n, ld, generator=g, device="cuda").bfloat16()[:, :k]
    return x, (torch.randn(o, k, generator=g, device="cuda") * k ** -0.5).bfloat16(), torch.randn(o, generator=g, device="cuda").bfloat16(), torch.randn(n, o, generator=g, device="cuda").bfloat16()


# tiles of 64 x 64 (up to 256 of them), 64 x 128, 128 x 128 and two of those per CU; depths below a stage, of one to five stages, with and without a rest; columns that end within a lane's eight
SIZES = [(65, 8, 64), (70, 64, 72), (1000, 72, 1000), (1024, 128, 1024), (1025, 192, 1024), (130, 264, 8192), (2047, 320, 1016), (2049, 256, 1500), (600, 1024, 5121), (2300, 136, 2600), (1196, 1024, 4096), (2304, 56, 3000), (450, 4096, 1102)]


@pytest.mark.parametrize("n,k,o", SIZES)
@pytest.mark.parametrize("bias", [False, True])
def test_products(n, k, o, bias):
    from jacobiforcing_amd import _native as N
    from jacobiforcing_amd import layer_ops as LO
    assert LO.linear_mid(n, k, o, torch.bfloat16)
    x, w, b, _ = _operands(n, k, o, k + 8, n + k + o)
    want = x.double() @ w.double().t() + (b.double() if bias else 0.0)
    st = LO._stream(x.device)
    for mode, dt in ((0, torch.bfloat16), (1, torch.float32), (2, torch.float32)):
        guard = torch.full((n + 1, o), 7.0, dtype=dt, device="cuda")
        N.check_layers(N.layers().jl_linear_mid(x.data_ptr(), N.JL_BF16, n, x.stride(0), w.data_ptr(), k, o, b.data_ptr() if bias else None, guard.data_ptr(), o, mode, st), "jl_linear_mid")
        got = guard[:n].double()
        assert bool((guard[n] == 7.0).all())
        # float sums of k products: a few 2 ** -24 of their size per product at most; results rounded to bfloat16, 2 ** -9
        assert (got - want).norm() <= (2.0 ** -8 if mode != 1 else 2.0 ** -24 * max(8, k ** 0.5)) * want.norm(), mode
        if mode == 2:
            assert torch.equal(guard[:n], guard[:n].bfloat16().float())
    assert torch.equal(LO.linear(x, w, b if bias else None).float(), guard[:n])      # the wrapper's way there: the same sums


@pytest.mark.parametrize("n,k,o", [(1, 64, 64), (70, 72, 72), (1025, 192, 1024), (600, 1024, 1021), (2049, 256, 1504), (1196, 2048, 4096), (300, 8192, 64)])
def test_products_onto_what_is_there(n, k, o):
    from jacobiforcing_amd import layer_ops as LO
    x, w, _, c = _operands(n, k, o, k + 16, n + o)
    want, got = c.double() + x.double() @ w.double().t(), c.clone()
    assert LO.linear_add_(got, x, w) is got
    assert (got.double() - want).norm() <= 2.0 ** -8 * want.norm()
    assert (got.double() - want).abs().max() <= (2.0 ** -8 + 2.0 ** -20) * want.abs().max()


# the same tiles with a unit in the epilogue: gates and linear branches of fewer columns than a tile's half, beside fours, and of every tile size
@pytest.mark.parametrize("n,k,f", [(65, 8, 32), (70, 64, 36), (1000, 72, 501), (1025, 192, 512), (130, 264, 4100), (2047, 320, 508), (600, 1024, 2562), (2300, 136, 1300), (2048, 1024, 2048)])
@pytest.mark.parametrize("kind", [0, 1, 2, 3])
def test_units(n, k, f, kind):
    from jacobiforcing_amd import layer_ops as LO
    x, w, _, _ = _operands(n, k, 2 * f, k + 8, n + k + f)
    got = LO.linear_gated(x, w, kind, 1.5, 1.25, 0.5)
    z = (x.double() @ w.double().t()).float()
    want = LO.gated_act(z, 0, f, f, kind, 1.5, 1.25, 0.5).double()     # the unit in 32 bits
    assert got.shape == (n, f) and got.dtype == torch.bfloat16
    # the sums as above, which a unit of slope up to two takes on; rounded once, 2 ** -9 of each at most
    assert (got.double() - want).norm() <= 2.0 ** -8 * want.norm() and (got.double() - want).abs().max() <= 2.0 ** -8 * want.abs().max()


def test_which_calls_the_library_keeps(monkeypatch):
    """Sizes beyond the rule, autocast, other types, operands that share memory with the result: the library's product, as before."""
    from jacobiforcing_amd import _native as N
    from jacobiforcing_amd import layer_ops as LO
    x, w, b, c = _operands(1500, 512, 1024, 512, 3)
    H, L = LO._host(), LO.linear_mid
    assert L(1500, 512, 1024, torch.bfloat16) == 2 and L(1500, 2048, 2048, torch.bfloat16) == 1 and L(8192, 2048, 2048, torch.bfloat16) == 0 and L(100, 4864, 896, torch.bfloat16) == 0 and L(9, 9, 9, torch.float16) == 0
    big, wide = torch.randn(1500, 2048, device="cuda").bfloat16(), torch.randn(2048, 2048, device="cuda").bfloat16()
    assert H.linear(big, wide, None, None) is not NotImplemented
    with torch.autocast("cuda", dtype=torch.float16):
        assert H.linear(big, wide, None, None) is NotImplemented and LO.linear(big, wide).dtype == torch.float16
        assert H.linear_add(c, x, w) is NotImplemented
    assert LO.linear_gated(x.half(), w.half(), 2) is None and LO.linear_gated(x, w[:1023], 2) is None and LO.linear_gated(x[:4], w, 2) is None
    assert H.linear_add(c, x.half(), w) is NotImplemented and H.linear_add(c[:, :512], x, w) is NotImplemented and H.linear_add(c, x, w[:, :256]) is NotImplemented
    square = torch.randn(64, 64, device="cuda").bfloat16()
    assert H.linear_add(square, square, square.clone()) is NotImplemented
    leaf = torch.randn(1024, 512, device="cuda").bfloat16().requires_grad_()
    assert H.linear_add(c, x, leaf) is NotImplemented


def test_a_sum_in_place_is_seen():
    """A result that a graph has kept, and one made under inference mode: as the library's product in place has it."""
    from jacobiforcing_amd import layer_ops as LO
    x, w, _, c = _operands(128, 64, 64, 64, 7)
    leaf = torch.ones(128, 64, device="cuda").bfloat16().requires_grad_()
    kept = (leaf * c).sum()
    assert LO._host().linear_add(c, x, w) is not NotImplemented
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        kept.backward()
    with torch.inference_mode():
        made = torch.zeros(128, 64, device="cuda", dtype=torch.bfloat16)
        assert LO._host().linear_add(made, x, w) is not NotImplemented
    assert LO._host().linear_add(made, x, w) is NotImplemented


def test_where_the_launch_is_the_better_one():
    from jacobiforcing_amd import _native as N
    ok = N.layers().jl_linear_mid_ok
    for want, sizes in ((2, ((1500, 512, 1024), (8192, 1024, 256), (8192, 2048, 64), (2048, 2048, 512))),
                        (1, ((2304, 1024, 2048), (2048, 1024, 4096), (1024, 2048, 4096), (2048, 2048, 2048), (300, 4096, 1024), (512, 4096, 2048))),
                        (0, ((2305, 1536, 1024), (700, 2048, 6144), (2048, 1536, 3072), (2048, 1024, 4097), (700, 4096, 2048), (512, 4096, 512), (299, 4096, 2048), (512, 4104, 2048), (256, 2048, 32000)))):
        for n, k, o in sizes:
            assert ok(n, k, o) == want, (n, k, o)
