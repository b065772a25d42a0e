"""Products of floats in three bfloat16 terms per operand, at the edges of their tiles and stages, against 64 bits, and with values that are not finite."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _close(got, want, size, K):
    # six products of terms per 16 depths are added in 32 bits, each sum rounded once; what is left out of a product is at most 2^-23 of it
    return bool(((got.double() - want).abs() <= ((6 * K / 16 + 32) * 2.0 ** -24 + 2.0 ** -22) * size).all())


@pytest.mark.parametrize("N,K,O,bias", [(65, 4, 12300, True), (129, 36, 8193, False), (1000, 28, 1537, True), (640, 64, 2500, True), (1281, 100, 1900, False), (2049, 1028, 1153, True), (96, 260, 20000, False)])
def test_linear(N, K, O, bias):
    from jacobiforcing_amd import layer_ops as LO
    dev = "cuda"
    assert LO.linear_split(N, K, O) and not LO.linear_small(N, K, O, 4)
    g = torch.Generator(device=dev).manual_seed(N + K + O)
    x = torch.randn(N, K + 12, generator=g, device=dev)[:, 8:8 + K]
    x = x * torch.logspace(-6, 6, N, device=dev).view(N, 1)
    w, b = torch.randn(O, K, generator=g, device=dev), torch.randn(O, generator=g, device=dev) if bias else None
    x = torch.cat([x, x], 1)[:, :K]                                                          # rows apart
    want = x.double() @ w.double().T + (b.double() if bias else 0)
    size = x.double().abs() @ w.double().abs().T + (b.double().abs() if bias else 0)
    for float_out in (None, True, False):
        got = LO.linear(x, w, b, float_out)
        assert got.dtype == torch.float32 and got.shape == (N, O) and _close(got, want, size, K)
    x = x.bfloat16()                                                                         # counts as float beside float weights
    assert _close(LO.linear(x, w, b, True), x.double() @ w.double().T + (b.double() if bias else 0), x.double().abs() @ w.double().abs().T + (b.double().abs() if bias else 0), K)


@pytest.mark.parametrize("N,K,O", [(700, 40, 2304), (1500, 68, 1536)])
def test_values_that_are_not_finite(N, K, O):
    """Infinities, NaN and overflowing sums come out as the float products have them; rows and columns without them are unchanged."""
    from jacobiforcing_amd import layer_ops as LO
    dev = "cuda"
    g = torch.Generator(device=dev).manual_seed(5)
    x, w = torch.randn(N, K, generator=g, device=dev), torch.randn(O, K, generator=g, device=dev)
    w[:, 7] = torch.where(w[:, 7] == 0, 1.0, w[:, 7]).bfloat16().float()                      # exact in one term: the others are zero
    clean = LO.linear(x, w)
    y, v = x.clone(), w.clone()
    y[3, 7], y[N - 1, 7], y[200, K - 1], y[300, 0] = float("inf"), -float("inf"), float("nan"), 3.4e38
    v[O - 1, 5] = float("inf")
    got, want = LO.linear(y, v), (y.double() @ v.double().T)
    want = torch.where(want.abs() > torch.finfo(torch.float32).max, want.sign() * float("inf"), want)
    rows, cols = [3, 200, 300, N - 1], [O - 1]
    for r in rows:
        assert torch.equal(got[r].isnan(), want[r].isnan()) and torch.equal(got[r].isinf(), want[r].isinf()) and torch.equal(got[r][got[r].isinf()].double(), want[r][want[r].isinf()])
    assert torch.equal(got[:, O - 1].isnan(), want[:, O - 1].isnan())
    rest = torch.ones(N, O, dtype=torch.bool, device=dev)
    rest[rows], rest[:, cols] = False, False
    assert bool(((got - clean).abs()[rest] <= (K + 64) * 2.0 ** -24 * (x.abs() @ w.abs().T)[rest]).all())


@pytest.mark.parametrize("low", [-110, -118, -122, -126, -130])
def test_the_smallest_operands(low):
    """Operands near float's end, against large ones: their terms end with bfloat16's last place, 2^-133, so half of it is lost of each, and nothing that shows from 2^-118 on."""
    from jacobiforcing_amd import layer_ops as LO
    dev, N, K, O = "cuda", 640, 512, 4096
    assert LO.linear_split(N, K, O)
    g = torch.Generator(device=dev).manual_seed(1)
    x, w = (torch.rand(N, K, generator=g, device=dev) + 1) * 2.0 ** low, (torch.rand(O, K, generator=g, device=dev) + 1) * 2.0 ** 90
    got, want = LO.linear(x, w).double(), x.double() @ w.double().T                           # all of one sign: a product's size is its value
    lost = 2.0 ** -134 * w.double().sum(1)
    assert bool(((got - want).abs() <= lost + ((6 * K / 16 + 32) * 2.0 ** -24 + 2.0 ** -22) * want).all())
    if low >= -118:
        # (-118: 2^-134 of 2^-118 is 2^-16 of an operand at most, and a mean of K of them, of either sign, 2^-20)
        assert float((got - want).norm() / want.norm()) <= 2.0 ** -19


def _lean(got, want):
    """The mean error against the values' root mean square, and what chance makes of it."""
    e = (got.double() - want) / want.pow(2).mean().sqrt()
    return float(e.mean().abs()), 5 * float(e.std()) / e.numel() ** 0.5


# the instructions cut sums towards minus infinity: by 2^-27 of them at a depth of 96, 2^-22 at 4096, were they not held with either sign in turn, which leaves a step's cut against its neighbour's
@pytest.mark.parametrize("N,K,O", [(4096, 96, 4096), (4096, 320, 4096), (6000, 832, 608), (2553, 2048, 3072), (4096, 4096, 4096), (640, 1100, 4096)])
def test_sums_lean_neither_way(N, K, O):
    from jacobiforcing_amd import layer_ops as LO
    assert LO.linear_split(N, K, O)
    g = torch.Generator(device="cuda").manual_seed(K)
    x, w = torch.randn(N, K, generator=g, device="cuda"), torch.randn(O, K, generator=g, device="cuda")
    lean, chance = _lean(LO.linear(x, w), x.double() @ w.double().T)
    assert lean <= 2.0 ** -28 + chance, lean


@pytest.mark.parametrize("n,W,ff,E", [(4000, 1024, 1024, 4), (3200, 1028, 516, 12)])
def test_experts_sums_lean_neither_way(n, W, ff, E):
    """The way down, in parts of 128 rows and tiles of 64 (what the way up leans by meets weights of either sign)."""
    from jacobiforcing_amd import _native as N, layer_ops as LO
    assert N.layers().jl_moe_float_tiles(n, E, W, ff) == (256 if n >= 320 * E else 64) and N.layers().jl_moe_tile_rows(N.JL_F32, n, E, W, ff) == 64
    g = torch.Generator(device="cuda").manual_seed(ff)
    h, logits = torch.randn(n, W, generator=g, device="cuda"), torch.randn(n, E, generator=g, device="cuda")
    up, down = torch.randn(E, ff, W, generator=g, device="cuda") * W ** -0.5, torch.randn(E, W, ff, generator=g, device="cuda") * ff ** -0.5
    got, want = LO.moe_experts(h, logits, None, 1, 1.0, up, down, route="top_softmax")[:, 0], torch.zeros(n, W, dtype=torch.float64, device="cuda")
    ids = logits.argmax(-1)
    for e in range(E):
        r = (ids == e).nonzero()[:, 0]
        want[r] = torch.relu(h[r].double() @ up[e].double().T) ** 2 @ down[e].double().T
    lean, chance = _lean(got, want)
    assert lean <= 2.0 ** -28 + chance, lean


@pytest.mark.parametrize("n,W,ff,E,top,gated,bad", [(1700, 36, 2052, 10, 2, True, False), (3300, 2060, 100, 4, 1, False, False), (3500, 1024, 520, 6, 1, True, True), (800, 1028, 516, 12, 4, True, True),
                                                     (705, 516, 1028, 6, 4, False, True)])
def test_experts(n, W, ff, E, top, gated, bad):
    """Experts of floats in tiles of 64 rows (fewer than 320 per expert) and parts of 128; a row that is not finite spoils no other."""
    from jacobiforcing_amd import _native as N, layer_ops as LO
    dev = "cuda"
    L = N.layers()
    tiles = L.jl_moe_float_tiles(n * top, E, W, ff)
    assert tiles == (256 if n * top >= 320 * E else 64) and L.jl_moe_tile_rows(N.JL_F32, n * top, E, W, ff) == 64
    g = torch.Generator(device=dev).manual_seed(n)
    h, logits = torch.randn(n, W, generator=g, device=dev), torch.randn(n, E, generator=g, device=dev)
    logits[:, 0] += 1.5                                                                       # uneven experts
    up, down = torch.randn(E, ff * (2 if gated else 1), W, generator=g, device=dev) * W ** -0.5, torch.randn(E, W, ff, generator=g, device=dev) * ff ** -0.5
    if bad:
        h[11, 3], h[n - 1, 0] = float("inf"), float("nan")
    got = LO.moe_experts(h, logits, None, top, 1.0, up, down, route="top_softmax", gated=(N.JL_ACT_SILU, 0.0, 1.0, 0.0) if gated else None)
    lead, ids = logits.double().topk(top, -1)
    p, want = lead.softmax(-1), torch.zeros(n, top, W, dtype=torch.float64, device=dev)
    size = torch.zeros_like(want)
    for e in range(E):
        r, c = (ids == e).nonzero(as_tuple=True)
        z = h[r].double() @ up[e].double().T
        z = torch.nn.functional.silu(z[:, :ff]) * z[:, ff:] if gated else torch.relu(z) ** 2
        want[r, c], size[r, c] = (z @ down[e].double().T) * p[r, c][:, None], (z.abs() @ down[e].double().abs().T) * p[r, c][:, None]
    fine = torch.ones(n, dtype=torch.bool, device=dev)
    if bad:
        fine[11], fine[n - 1] = False, False
        assert not bool(got[11].isfinite().any()) and (not gated or bool(got[n - 1].isnan().all()))      # relu's square of NaN is zero
    # the units carry the way up's error ((6 W / 16 + 32) roundings of sums about sqrt(W) times their size, twice for a product or a square) into every term of the way down
    tol = ((6 * ff / 16 + 64) * 2.0 ** -24 + 2.0 ** -21) * size + 4 * (6 * W / 16 + 32) * 2.0 ** -24 * size.amax(-1, keepdim=True)
    assert bool(((got.double() - want).abs() <= tol)[fine].all())
