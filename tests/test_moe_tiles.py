"""Routed experts at the edges of the grouped products' tiles (32, 64 and 128 rows, columns and depths beside their multiples), against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("N,E,top,W,ff,gated,identity,skew", [
    (1, 3, 2, 8, 8, True, 0, 0.0), (33, 4, 4, 64, 40, False, 0, 0.0), (130, 16, 2, 72, 136, True, 3, 0.0), (70, 5, 2, 200, 60, True, 0, 0.0), (97, 4, 1, 1000, 24, False, 2, 0.0),
    (300, 2, 1, 264, 264, True, 0, 0.0), (1025, 7, 3, 128, 520, False, 0, 3.0), (700, 300, 2, 96, 32, True, 9, 0.0), (513, 4, 2, 36, 68, True, 0, 9.0), (50, 4, 2, 30, 50, True, 0, 0.0),
    (5000, 4000, 4, 32, 16, False, 96, 0.0),
])
def test_experts(dtype, N, E, top, W, ff, gated, identity, skew):
    """``skew``: how much the router prefers the first expert (its tiles many, others' few or none)."""
    from jacobiforcing_amd import layer_ops as LO
    dev, dt = "cuda", getattr(torch, dtype)
    g = torch.Generator(device=dev).manual_seed(N + E)
    rnd = lambda *s, std=1.0: (torch.randn(*s, generator=g, device=dev) * std).to(dt)
    h, z = rnd(N, W), torch.randn(N, E + identity, generator=g, device=dev)
    z[:, 0] += skew
    up, down = rnd(E, 2 * ff if gated else ff, W, std=W ** -0.5), rnd(E, W, ff, std=ff ** -0.5)
    got = LO.moe_experts(h, z, None, top, 1.0, up, down, route="top_softmax", gated=(LO.ACT_SILU, 0.0, 1.0, 0.0) if gated else None, identity=identity)
    y, ids = (got[0], got[1]) if identity else (got, None)
    val, idx = torch.sort(z, dim=-1, descending=True, stable=True)
    idx, wt = idx[:, :top], torch.softmax(val[:, :top].double(), -1)
    if ids is not None:
        assert torch.equal(ids.long(), idx)
    want, real = torch.zeros(N, top, W, dtype=torch.float64, device=dev), idx < E
    for e in idx[real].unique().tolist():
        n, s = (idx == e).nonzero(as_tuple=True)
        u = h[n].double() @ up[e].double().T
        a = torch.nn.functional.silu(u[:, :ff]) * u[:, ff:] if gated else torch.relu(u) ** 2
        a = a.to(dt).double()                             # the units are stored in the activations' dtype
        want[n, s] = (a @ down[e].double().T) * wt[n, s].unsqueeze(-1)
    err = (y.double() - want)[real]
    # float: sums of K products rounded one by one, 2 ** -24 each, in two products; bfloat16: the units may round the other way (2 ** -8 of each, averaged by the sum)
    tol = (W + ff) ** 0.5 * 2.0 ** -22 if dtype == "float32" else 2.0 ** -8
    assert err.norm() <= tol * want.norm() and err.abs().max() <= 16 * tol * want.abs().max()
