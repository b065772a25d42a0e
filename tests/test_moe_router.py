"""The experts' router product, choice and grouping in one call: the same choices, weights and outputs, bit for bit, as from logits handed in.  Operands are small whole numbers, so that every
order of the sums is exact and ties are many."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def run(monkeypatch, N, K, E, identity, top, x_dtype, bias, route, pad=0, gated=False):
    from jacobiforcing_amd import layer_ops as LO
    for limit in ("ROUTER_DEPTH", "ROUTER_DEPTH_FEW"):                         # also where a product of its own is the faster one
        monkeypatch.setattr(LO, limit, 1 << 30)
    g = torch.Generator(device="cuda").manual_seed(N + K + E)
    whole = lambda lim, *s: torch.randint(-lim, lim + 1, s, generator=g, device="cuda")
    Er, W, ff = E + identity, 64, 32
    x = whole(4, N, K + pad).to(x_dtype)[:, :K]
    w = (whole(4, Er, K) / 256).float()                                        # K * 16 / 256 in steps of 1 / 256: exact in 24 bits
    b = (whole(8, Er) / 16).float() if bias else None
    corr = (whole(8, Er) / 32).float() if route != "top_softmax" else None
    h = torch.randn(N, W, generator=g, device="cuda").bfloat16()
    up, down = torch.randn(E, (2 if gated else 1) * ff, W, generator=g, device="cuda").bfloat16(), torch.randn(E, W, ff, generator=g, device="cuda").bfloat16()
    logits = x.double() @ w.double().T
    logits = (logits if b is None else logits + b.double()).float()
    kw = dict(route=route, renorm_eps=1e-20, identity=identity, gated=(LO.ACT_SILU, 0.0, 1.0, 0.0) if gated else None)
    with monkeypatch.context() as m:
        m.setattr(LO, "ROUTER_OUTPUTS", 0)                                     # choice and grouping in launches of their own
        want = LO.moe_experts(h, logits, corr, top, 0.5, up, down, **kw)
    for got in (LO.moe_experts(h, logits, corr, top, 0.5, up, down, **kw), LO.moe_experts(h, None, corr, top, 0.5, up, down, router=(x, w, b), **kw)):
        if not identity:
            assert torch.equal(got, want)
            continue
        real = want[1] < E
        assert torch.equal(got[1], want[1]) and torch.equal(got[2], want[2]) and torch.equal(got[0][real], want[0][real])
    return LO._router_in_one(x, w, b)


@pytest.mark.parametrize("x_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,K,E,identity,top,bias,route,pad", [
    (1, 64, 1, 0, 1, False, "sigmoid", 0), (16, 1024, 16, 0, 4, True, "top_softmax", 0), (17, 2048, 17, 5, 3, False, "softmax_renorm", 8), (32, 36, 33, 7, 4, True, "softmax_renorm", 28),
    (33, 512, 48, 16, 8, False, "sigmoid", 0), (64, 4, 7, 1, 2, True, "top_softmax", 4), (1000, 200, 9, 0, 9, False, "softmax_renorm", 0), (4097, 1032, 32, 0, 4, True, "top_softmax", 0),
    (8192, 128, 24, 6, 4, False, "sigmoid", 0), (16384, 32, 64, 0, 2, False, "softmax_renorm", 0), (40, 64, 3, 61, 64, False, "softmax_renorm", 0),
])
def test_the_same_as_from_logits(monkeypatch, x_dtype, N, K, E, identity, top, bias, route, pad):
    """One workgroup and many, one to four blocks of outputs, depths beside whole lines, rows apart, experts without rows, choices of all outputs."""
    assert run(monkeypatch, N, K, E, identity, top, x_dtype, bias, route, pad), "the launches did not run"


@pytest.mark.parametrize("x_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,K,E,identity,top,bias,route,pad", [(1, 2048, 16, 0, 4, True, "sigmoid", 0), (16, 516, 60, 4, 3, False, "top_softmax", 4), (17, 2052, 17, 0, 2, True, "softmax_renorm", 12),
                                                               (65, 1028, 30, 9, 4, True, "sigmoid", 12), (2048, 1032, 20, 0, 4, False, "softmax_renorm", 0), (2049, 1024, 32, 0, 4, False, "sigmoid", 0)])
def test_products_in_slices_of_the_depth(monkeypatch, x_dtype, N, K, E, identity, top, bias, route, pad):
    """The smallest products that are sliced, depths whose slices end beside whole lines, one workgroup and the most (one more: whole)."""
    from jacobiforcing_amd import _native as N_
    assert N_.layers().jl_moe_router_slices(N, E + identity, K) == (4 if N <= 2048 else 1)
    assert run(monkeypatch, N, K, E, identity, top, x_dtype, bias, route, pad), "the launches did not run"


@pytest.mark.parametrize("N,K,E", [(16385, 16, 4), (20, 30, 8), (50, 64, 65)])
def test_what_the_launches_do_not_take(monkeypatch, N, K, E):
    """More tokens, depths beside 16-byte borders, more outputs: the product, the choice and the grouping one after the other."""
    assert not run(monkeypatch, N, K, E, 0, 2, torch.float32, True, "top_softmax")


@pytest.mark.parametrize("route", ["sigmoid", "softmax_renorm", "top_softmax"])
def test_logits_that_are_not_finite(monkeypatch, route):
    """Infinities are chosen (or not) as before; a token with one that is not a number shows it in its outputs, and no other token does."""
    from jacobiforcing_amd import layer_ops as LO
    g = torch.Generator(device="cuda").manual_seed(3)
    N, E, W, ff = 70, 6, 64, 32
    h, up, down = (torch.randn(*s, generator=g, device="cuda").bfloat16() for s in ((N, W), (E, ff, W), (E, W, ff)))
    z = torch.randn(N, E, generator=g, device="cuda")
    z[3, 2], z[4, 1], z[5] = float("inf"), -float("inf"), -float("inf")
    with monkeypatch.context() as m:
        m.setattr(LO, "ROUTER_OUTPUTS", 0)
        want = LO.moe_experts(h, z, None, 2, 1.0, up, down, route=route)
    assert torch.equal(LO.moe_experts(h, z, None, 2, 1.0, up, down, route=route).nan_to_num(7.0), want.nan_to_num(7.0))
    z[9, 4] = float("nan")
    y = LO.moe_experts(h, z, None, 2, 1.0, up, down, route=route)
    assert y[9].isnan().any() and torch.equal(torch.cat([y[:9], y[10:]]).nan_to_num(7.0), torch.cat([want[:9], want[10:]]).nan_to_num(7.0))


@pytest.mark.parametrize("n,K,E,dtype,one", [(32, 2048, 48, "float32", True), (512, 2048, 49, "bfloat16", False), (513, 2048, 16, "float32", True), (513, 1028, 17, "float32", False), (2048, 1024, 48, "bfloat16", True), (2048, 1024, 64, "bfloat16", False),
                                             (8192, 2048, 32, "float32", False), (8192, 3072, 64, "bfloat16", True)])
def test_where_the_product_is_in_the_launch(n, K, E, dtype, one):
    """Up to a product of depth and blocks of 16 outputs that grows with the tokens in 16 bits; beyond, the same choices from ``linear``'s logits."""
    from jacobiforcing_amd import layer_ops as LO
    x, w = torch.zeros(n, K, device="cuda", dtype=getattr(torch, dtype)), torch.zeros(E, K, device="cuda")
    assert LO._router_operands(x, w, None) and LO._router_in_one(x, w, None) == one


@pytest.mark.parametrize("route", ["sigmoid", "softmax_renorm", "top_softmax"])
@pytest.mark.parametrize("E,correct", [(6, False), (6, True), (64, True)])
def test_choices_among_values_that_are_not_numbers(monkeypatch, route, E, correct):
    """... count as the largest, ties to the lowest index, whichever launches make the choice (how many tokens a step has decides that)."""
    from jacobiforcing_amd import layer_ops as LO
    g = torch.Generator(device="cuda").manual_seed(E)
    N, W, ff, nan = 70, 64, 32, float("nan")
    h, up, down = (torch.randn(*s, generator=g, device="cuda").bfloat16() for s in ((N, W), (E - 1, ff, W), (E - 1, W, ff)))
    z, corr = torch.randn(N, E, generator=g, device="cuda"), torch.randn(E, generator=g, device="cuda") if correct else None
    z[2, 4], z[3, [1, E - 1]], z[4], z[5, 2:], z[6, 3], z[6, 1] = nan, nan, nan, nan, float("inf"), nan
    run = lambda: LO.moe_experts(h, z, corr, 3, 1.0, up, down, route=route, identity=1)
    got = run()
    monkeypatch.setattr(LO, "ROUTER_OUTPUTS", 0)
    want = run()
    assert torch.equal(got[1], want[1]) and torch.equal(got[2].nan_to_num(7.0), want[2].nan_to_num(7.0))
    first = [[4], [1, E - 1], [0, 1, 2], [2, 3, 4]]
    if route == "top_softmax" or (route == "sigmoid" and not correct):
        assert all(want[1][2 + i, :len(f)].tolist() == f for i, f in enumerate(first))
    assert all(len(set(row)) == 3 for row in want[1].tolist())


@pytest.mark.parametrize("x_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,K,E", [(1, 1024, 16), (32, 2048, 33), (70, 520, 64), (2000, 200, 9)])
def test_weights_of_random_operands(monkeypatch, x_dtype, N, K, E):
    """The product's operands and sums keep 32 bits: every output's weight against 64 bits.  A rounding (2 ** -24) of each product and of its sums comes to less than 1e-6 of a logit of size one; a
    weight rounded to 16 bits would be off by 2 ** -9, which is 3e-4 in a sigmoid."""
    from jacobiforcing_amd import layer_ops as LO
    for limit in ("ROUTER_DEPTH", "ROUTER_DEPTH_FEW"):
        monkeypatch.setattr(LO, limit, 1 << 30)
    g = torch.Generator(device="cuda").manual_seed(N + E)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, w, b, corr = rnd(N, K).to(x_dtype), rnd(E, K) * K ** -0.5, rnd(E), rnd(E)
    h, up, down = rnd(N, 64).bfloat16(), rnd(E - 1, 32, 64).bfloat16(), rnd(E - 1, 64, 32).bfloat16()
    assert LO._router_in_one(x, w, b)
    z = x.double() @ w.double().T + b.double()
    for route, want in (("sigmoid", z.sigmoid()), ("softmax_renorm", z.softmax(1)), ("top_softmax", z.softmax(1))):
        _, ids, weights = LO.moe_experts(h, None, corr, E, 1.0, up, down, route=route, identity=1, router=(x, w, b))
        assert torch.equal(ids.sort(1).values, torch.arange(E, device="cuda", dtype=torch.int32).expand(N, E))
        got = torch.zeros_like(z).scatter_(1, ids.long(), weights.double())
        assert float((got - want).abs().max()) < 2e-6, route
