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


@pytest.mark.parametrize("dtype,K,gated", [("bfloat16", 1032, True), ("bfloat16", 2048, False), ("float32", 516, True), ("float32", 1028, False)])
@pytest.mark.parametrize("tile", [32, 64, 128])
@pytest.mark.parametrize("far", ["rows gathered from", "rows in order", "weights"])
def test_operands_beyond_4_gib(dtype, K, gated, tile, far):
    """The tiles of the matrix instructions reach them, in the same order of sums: bit for bit what the same rows give as a small product."""
    from jacobiforcing_amd import _native as N
    from jacobiforcing_amd import layer_ops as LO
    if dtype == "float32" and tile == 128:
        pytest.skip("float tiles have up to 64 rows")
    dev, dt, lib, E, n_out = "cuda", getattr(torch, dtype), N.layers(), 2, 24
    size, code, st = dt.itemsize, LO._code(dt), torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device=dev).manual_seed(K)
    rows, beyond = 300, (1 << 32) // (K * size) + 5                  # rows of 32 bits' reach and five more
    mode = 1 if far == "rows in order" else N.JL_MOE_UP_PLAIN
    if far == "weights":
        if gated:
            pytest.skip("one product's columns reach as far")
        X, W, cols = torch.randn(rows, K, generator=g, device=dev).to(dt), torch.zeros(E, beyond + n_out, K, dtype=dt, device=dev), beyond + n_out
        W[:, -n_out:] = torch.randn(E, n_out, K, generator=g, device=dev).to(dt)
    else:
        X, W, cols = torch.zeros(beyond + rows, K, dtype=dt, device=dev), torch.randn(E, (2 if gated and mode != 1 else 1) * n_out, K, generator=g, device=dev).to(dt), n_out
        X[-rows:] = torch.randn(rows, K, generator=g, device=dev).to(dt)

    def run(x, w, n_cols, first_row):
        """Expert 0 has 170 of the 300 rows, expert 1 the others; gathered backwards, or in order from ``first_row`` on."""
        total = x.shape[0]
        perm = torch.arange(total - 1, total - 1 - rows, -1, dtype=torch.int32, device=dev) if mode != 1 else torch.arange(first_row + rows, dtype=torch.int32, device=dev)
        start = 0 if mode != 1 else first_row
        t_e, t_r = [], []
        for e, (lo, hi) in enumerate(((start, start + 170), (start + 170, start + 300))):
            t_e += [e] * len(range(lo, hi, tile))
            t_r += list(range(lo, hi, tile))
        offs = torch.tensor([start, start + 170, start + rows, len(t_e)], dtype=torch.int32, device=dev)
        count = total // tile + E if mode != 1 else len(t_e)          # as many tiles as a step of all rows would have: the launch goes by it
        te, tr = torch.full((count,), -1, dtype=torch.int32, device=dev), torch.zeros(count, dtype=torch.int32, device=dev)
        te[:len(t_e)], tr[:len(t_e)] = torch.tensor(t_e, device=dev), torch.tensor(t_r, device=dev)
        out = torch.empty(start + rows, n_cols, dtype=torch.float32 if mode == 1 else dt, device=dev)
        wts = torch.ones(start + rows, device=dev)
        if gated and mode != 1:
            rc = lib.jl_moe_gemm_gated(x.data_ptr(), w.data_ptr(), code, K, n_cols, 1, perm.data_ptr(), offs.data_ptr(), te.data_ptr(), tr.data_ptr(), count, E, tile, N.JL_ACT_SILU, 0.0, 1.0,
                                       0.0, out.data_ptr(), st)
        else:
            rc = lib.jl_moe_gemm(x.data_ptr(), w.data_ptr(), code, mode, K, n_cols, 1, perm.data_ptr(), offs.data_ptr(), te.data_ptr(), tr.data_ptr(), count, E, tile,
                                 wts.data_ptr() if mode == 1 else None, out.data_ptr(), st)
        assert rc == 0
        return out[start:, -n_out:].clone()

    got = run(X, W, cols, X.shape[0] - rows)
    want = run(X[-rows:].contiguous(), W[:, -n_out:].contiguous() if far == "weights" else W, n_out, 0)
    assert torch.equal(got, want) and bool(want.any())


def test_tile_heights_of_each_type():
    """Float rows never get the 128-row tiles, and asking for them is refused."""
    from jacobiforcing_amd import _native as N
    lib = N.layers()
    heights = {dt: {lib.jl_moe_tile_rows(dt, rows, E, W, ff) for rows in (4, 500, 5000, 100000) for E in (2, 16, 64) for W in (64, 1024, 4096) for ff in (64, 1024)} for dt in (N.JL_BF16, N.JL_F32)}
    assert heights[N.JL_BF16] == {32, 64, 128} and heights[N.JL_F32] == {32, 64}
    x, i = torch.zeros(64, 64, device="cuda"), torch.zeros(64, dtype=torch.int32, device="cuda")
    assert lib.jl_moe_gemm(x.data_ptr(), x.data_ptr(), N.JL_F32, N.JL_MOE_UP_PLAIN, 64, 64, 1, i.data_ptr(), i.data_ptr(), i.data_ptr(), i.data_ptr(), 1, 1, 128, None, x.data_ptr(), None) == -1


@pytest.mark.parametrize("dtype,tile", [("bfloat16", 32), ("bfloat16", 64), ("bfloat16", 128), ("float32", 32), ("float32", 64), ("float32", 256)])
@pytest.mark.parametrize("N,E,top,W,ff,gated,identity,skew", [
    (1, 3, 2, 8, 8, True, 0, 0.0), (130, 3, 2, 24, 32, True, 0, 0.0), (259, 4, 2, 64, 96, True, 1, 0.0), (257, 2, 1, 96, 64, False, 0, 0.0), (300, 5, 2, 72, 264, True, 0, 0.0), (200, 3, 1, 64, 50, True, 0, 0.0),
    (513, 9, 1, 160, 136, False, 0, 9.0), (1100, 2, 1, 520, 264, True, 0, 1.0), (640, 40, 2, 40, 256, True, 4, 3.0), (385, 4, 3, 1024, 520, True, 0, 0.0),
])
def test_every_tile_height(monkeypatch, dtype, tile, N, E, top, W, ff, gated, identity, skew):
    """The same with tiles of one height: depths of one, two, three and more stages, beside and below them, columns beside their fours, experts with few rows, many or none."""
    from jacobiforcing_amd import _native as N_, layer_ops as LO
    lib, host, launched = N_.layers(), LO._host(), []
    gemm = lib.jl_moe_gemm

    class Watched:
        def __getattr__(self, name):
            def call(*a):
                r = getattr(host, name)(*a)
                if name == "moe_experts" and r is not NotImplemented:
                    launched.append(a[13])
                return r
            return call
    monkeypatch.setattr(lib, "jl_moe_tile_rows", lambda *a: 64 if (dtype, tile) == ("float32", 256) else tile, raising=False)
    monkeypatch.setattr(lib, "jl_moe_float_tiles", lambda *a: tile, raising=False)
    monkeypatch.setattr(lib, "jl_moe_tile_pairs", lambda *a: 0, raising=False)
    monkeypatch.setattr(lib, "jl_moe_gemm", lambda *a: launched.append(a[13]) or gemm(*a), raising=False)
    monkeypatch.setattr(LO, "_H", Watched())
    test_experts(dtype, N, E, top, W, ff, gated, identity, skew)
    assert launched and set(launched) == {tile}, launched


@pytest.mark.parametrize("dtype,tile,N,E,W,ff", [("bfloat16", 128, 4096, 16, 1024, 512), ("bfloat16", 64, 3000, 40, 520, 256), ("float32", 64, 2048, 16, 1024, 256)])
def test_tile_heights_that_the_rule_chooses(dtype, tile, N, E, W, ff):
    from jacobiforcing_amd import _native as N_
    from jacobiforcing_amd import layer_ops as LO
    assert N_.layers().jl_moe_tile_rows(LO._code(getattr(torch, dtype)), 4 * N, E, W, ff) == tile
    test_experts(dtype, N, E, 4, W, ff, True, 0, 0.0)
