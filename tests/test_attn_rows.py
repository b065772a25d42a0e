"""The 128-row attention tiles of long portions at the sizes where they can go wrong, against attention in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def reference(q, k, v, starts, counts, pages, page, H, G, Gv, D, Dv, scale, window, chunk, cap, sink):
    out, r0 = [], 0
    for s, n, tab in zip(starts, counts, pages):
        total = s + n
        tok = torch.tensor([tab[j // page] * page + j % page for j in range(total)], device=q.device)
        qq = q[r0:r0 + n].double().view(n, H, D).transpose(0, 1)
        kk = k[tok].double().view(total, G, D).transpose(0, 1).repeat_interleave(H // G, 0)
        vv = v[tok].double().view(total, Gv, Dv).transpose(0, 1)[torch.arange(H, device=q.device) // (H // G) % Gv]
        z = qq @ kk.transpose(1, 2) * scale
        if cap:
            z = cap * torch.tanh(z / cap)
        i, j = torch.arange(s, total, device=q.device).view(n, 1), torch.arange(total, device=q.device).view(1, total)
        see = j <= i
        if window:
            see = see & (i - j < window)
        if chunk:
            see = see & (i // chunk == j // chunk)
        z = z.masked_fill(~see, float("-inf"))
        if sink is not None:
            z = torch.cat([z, sink.double().view(H, 1, 1).expand(H, n, 1)], -1)
        w = torch.softmax(z, -1)[..., :total]
        out.append((w @ vv).transpose(0, 1).reshape(n, H * Dv))
        r0 += n
    return torch.cat(out)


# key and value widths at and beside the multiples of 64 (key rows in LDS) and 32 / 64 / 128 (value rows)
@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("H,G,Gv,D,Dv,window,chunk,cap,page,pad", [
    (16, 4, 4, 128, 128, 0, 0, 0.0, 64, 0), (16, 16, 16, 64, 64, 0, 0, 0.0, 64, 0), (16, 2, 2, 8, 32, 0, 0, 0.0, 64, 0), (24, 4, 4, 72, 96, 100, 0, 0.0, 64, 0),
    (16, 4, 2, 136, 64, 0, 0, 0.0, 48, 0), (20, 20, 20, 192, 128, 65, 0, 0.0, 64, 0), (40, 1, 1, 200, 96, 0, 0, 0.0, 64, 4), (16, 2, 2, 256, 128, 0, 0, 0.0, 64, 0),
    (16, 4, 4, 128, 128, 0, 100, 5.0, 64, 0), (16, 1, 0, 160, 128, 0, 0, 0.0, 64, 0), (16, 1, 0, 96, 64, 63, 0, 0.0, 64, 4), (33, 1, 0, 256, 32, 0, 64, 2.0, 40, 0),
])
def test_wide_tiles(dtype, H, G, Gv, D, Dv, window, chunk, cap, page, pad):
    """Unequal requests, two of them continuing inside a page; ``pad``: rows of the pools start at 8-byte borders only; Gv 0: the values are the key
    rows' first columns; pools hold NaN wherever nothing was written."""
    from jacobiforcing_amd import layer_ops as LO
    dev, dt = "cuda", getattr(torch, dtype)
    starts, counts = [0, 37, 1, 0], [-(-16384 * (1 if dtype == "bfloat16" else 2) // H), 131, 64, 33]
    g = torch.Generator(device=dev).manual_seed(D + H)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev).to(dt)
    need = [-(-(s + n) // page) for s, n in zip(starts, counts)]
    ids = torch.randperm(sum(need) + 3, generator=torch.Generator().manual_seed(H)).tolist()
    pages = [[ids.pop() for _ in range(n)] for n in need]
    tokens = (sum(need) + 3) * page
    nan = lambda width: torch.full((tokens, width), float("nan"), dtype=dt, device=dev)
    kp = nan(G * D + pad)
    k = kp[:, :G * D]
    v = k[:, :Dv] if Gv == 0 else nan(Gv * Dv + pad)[:, :Gv * Dv]
    for s, n, tab in zip(starts, counts, pages):
        tok = torch.tensor([tab[j // page] * page + j % page for j in range(s + n)], device=dev)
        k[tok] = rnd(s + n, G * D)
        if Gv:
            v[tok] = rnd(s + n, Gv * Dv)
    q, sink = rnd(sum(counts), H * D), torch.randn(H, generator=g, device=dev)
    batch = LO.RaggedBatch.build(counts, starts, [0, 1, 2, 3], pages, page, dev)
    gate = rnd(sum(counts), H)
    got = LO.attn_sweep(q, k, v, batch, H, G, D, Dv, D ** -0.5, window, value_heads=Gv, float_out=True, sink=sink, gate=gate, gate_per_head=True, chunk=chunk, softcap=cap)
    assert ("longest first", 128 // min(H // G, 32), None) in batch._tiles, "the 128-row form did not run"
    want = reference(q, k, v, starts, counts, pages, page, H, G, Gv or 1, D, Dv, D ** -0.5, window, chunk, cap, sink)
    want = (want.view(-1, H, Dv) * torch.sigmoid(gate.double()).unsqueeze(-1)).view_as(want)
    assert torch.isfinite(got).all()
    # weights are rounded to bfloat16 (2 ** -9 relative, independently): a sum of them is off by less than that of its largest terms; in float a score of
    # size 5 (sums of D products) is 2 ** -21 off and moves its weight by as much
    err, tol = (got.double() - want).abs(), 2.0 ** -8 if dtype == "bfloat16" else 2.0 ** -20
    assert err.max() < 2 * tol * want.abs().max() and err.norm() < tol * want.norm()


@pytest.mark.parametrize("H,G,Gv,D,Dv,window,chunk,cap,page", [
    (8, 2, 2, 128, 128, 0, 0, 0.0, 64), (3, 3, 3, 20, 32, 50, 0, 0.0, 32), (40, 1, 0, 160, 128, 0, 0, 0.0, 64), (12, 4, 2, 252, 96, 0, 128, 3.0, 48), (6, 1, 0, 68, 64, 300, 0, 0.0, 64),
])
def test_float_tiles_with_shared_out_keys(H, G, Gv, D, Dv, window, chunk, cap, page):
    """Decoded tokens and short portions in float: 32-row tiles whose keys several workgroups share."""
    from jacobiforcing_amd import layer_ops as LO
    dev, dt = "cuda", torch.float32
    starts, counts = [700, 0, 333, 1023, 64], [1, 1, 5, 1, 33]
    g = torch.Generator(device=dev).manual_seed(D + H)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    need = [-(-(s + n) // page) for s, n in zip(starts, counts)]
    ids = torch.randperm(sum(need) + 3, generator=torch.Generator().manual_seed(H)).tolist()
    pages = [[ids.pop() for _ in range(n)] for n in need]
    k = torch.full(((sum(need) + 3) * page, G * D), float("nan"), device=dev)
    v = k[:, :Dv] if Gv == 0 else torch.full((k.shape[0], Gv * Dv), float("nan"), device=dev)
    for s, n, tab in zip(starts, counts, pages):
        tok = torch.tensor([tab[j // page] * page + j % page for j in range(s + n)], device=dev)
        k[tok] = rnd(s + n, G * D)
        if Gv:
            v[tok] = rnd(s + n, Gv * Dv)
    q, sink, gate = rnd(sum(counts), H * D), rnd(H), rnd(sum(counts), H * Dv)
    batch = LO.RaggedBatch.build(counts, starts, list(range(5)), pages, page, dev)
    got = LO.attn_sweep(q, k, v, batch, H, G, D, Dv, D ** -0.5, window, value_heads=Gv, sink=sink, gate=gate, chunk=chunk, softcap=cap, out_scale=0.7)
    want = reference(q, k, v, starts, counts, pages, page, H, G, Gv or 1, D, Dv, D ** -0.5, window, chunk, cap, sink) * torch.sigmoid(gate.double()) * 0.7
    err = (got.double() - want).abs()
    assert torch.isfinite(got).all() and err.max() < 2.0 ** -19 * want.abs().max() and err.norm() < 2.0 ** -20 * want.norm()


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("H,D,R,rd,Dv,rot,pairing,window,gate,built", [
    (5, 64, 128, 32, 64, 32, "ROT_NEIGHBOURS", 0, None, (0, 1, 2, 3)), (16, 128, 512, 64, 128, 64, "ROT_HALVES", 100, "full", (0, 1, 2, 3)), (3, 8, 64, 8, 32, 4, "ROT_NEIGHBOURS", 1, "head", (1, 3)),
    (2, 248, 32, 8, 96, 8, "ROT_HALVES", 0, "full", (0,)), (4, 64, 96, 0, 128, 0, "ROT_HALVES", 37, "head", (0, 1, 3)), (33, 120, 40, 72, 64, 72, "ROT_NEIGHBOURS", 300, None, (1, 2)),
])
def test_latent_attention_with_built_keys(monkeypatch, dtype, H, D, R, rd, Dv, rot, pairing, window, gate, built):
    """Some or all requests of a step on keys and values built per head, the others over the latent; the last request brings one token."""
    from jacobiforcing_amd import layer_ops as LO
    dev, dt, page = "cuda", getattr(torch, dtype), 32
    monkeypatch.setattr(LO, "_latent_built_requests", lambda *a: list(built))
    starts, counts = [0, 45, 3, 200], [129, 300, 128, 1]
    g = torch.Generator(device=dev).manual_seed(H + R)
    rnd = lambda *s, std=1.0: (torch.randn(*s, generator=g, device=dev) * std).to(dt)
    need = [-(-(s + n) // page) for s, n in zip(starts, counts)]
    ids = torch.randperm(sum(need) + 2, generator=torch.Generator().manual_seed(H)).tolist()
    pages = [[ids.pop() for _ in range(n)] for n in need]
    pool = torch.full(((sum(need) + 2) * page, R + rd), float("nan"), dtype=dt, device=dev)
    for s, n, tab in zip(starts, counts, pages):
        pool[torch.tensor([tab[j // page] * page + j % page for j in range(s + n)], device=dev)] = rnd(s + n, R + rd)
    n = sum(counts)
    wide = rnd(n, H * (D + rd) + 8)                       # the queries are a column range of wider rows
    w_uk, w_uv, sink = rnd(H * D, R, std=R ** -0.5), rnd(H * Dv, R, std=R ** -0.5), torch.randn(H, generator=g, device=dev)
    gates = None if gate is None else rnd(n, H if gate == "head" else H * Dv)
    batch = LO.RaggedBatch.build(counts, starts, [0, 1, 2, 3], pages, page, dev)
    a = torch.arange(512, dtype=torch.float32, device=dev).view(-1, 1) * torch.rand(max(rot, 2) // 2, generator=g, device=dev).view(1, -1)
    cos, sin = (a.cos().contiguous(), a.sin().contiguous()) if rot else (None, None)
    q64 = wide[:, :H * (D + rd)].double().view(n, H, D + rd)
    tail = q64[..., D:D + rot]
    if rot:
        c, s = cos.double()[batch.pos.long()].unsqueeze(1), sin.double()[batch.pos.long()].unsqueeze(1)
        near = pairing == "ROT_NEIGHBOURS"
        u, v = (tail[..., 0::2], tail[..., 1::2]) if near else (tail[..., :rot // 2], tail[..., rot // 2:])
        x, y = u * c - v * s, v * c + u * s
        tail = torch.stack([x, y], -1).flatten(-2) if near else torch.cat([x, y], -1)
    q64 = torch.cat([q64[..., :D], tail, q64[..., D + rot:]], -1)
    lat = pool.double()
    k64 = torch.cat([(lat[:, :R] @ w_uk.double().T).view(-1, H, D), lat[:, R:].unsqueeze(1).expand(-1, H, rd)], -1).flatten(1)
    scale = (D + rd) ** -0.5
    want = reference(q64.flatten(1), k64, lat[:, :R] @ w_uv.double().T, starts, counts, pages, page, H, H, H, D + rd, Dv, scale, window, 0, 0.0, sink)
    if gate is not None:
        gg = torch.sigmoid(gates.double())
        want = want * (gg if gate == "full" else gg.repeat_interleave(Dv, 1))
    got = LO.latent_attention(wide[:, :H * (D + rd)], pool, torch.cat([w_uk, w_uv]), w_uk.view(H, D, R), w_uv.view(H, Dv, R).transpose(1, 2).contiguous(), batch, H, D, R, rd, Dv, rot, cos, sin,
                              getattr(LO, pairing), scale, window, sink=sink, gate=gates, gate_per_head=gate == "head")
    # queries, keys, values, weights and the result are rounded to bfloat16 once each (2 ** -9 relative); a score of size 3 moves its weight by 1.2 %
    err, tol = (got.double() - want).abs(), 2.0 ** -6 if dtype == "bfloat16" else 2.0 ** -19
    assert torch.isfinite(got).all() and err.norm() < tol * want.norm() and err.max() < 4 * tol * want.abs().max()


@pytest.mark.parametrize("dtype,single", [("bfloat16", False), ("float32", False), ("float32", True)])
def test_more_tiles_than_a_short_grid_axis_holds(dtype, single):
    """One portion in more than 65 535 tiles of 128 rows (``single``: as many decoding requests, tiles of 32 rows), as in two steps."""
    from jacobiforcing_amd import layer_ops as LO
    dev, dt, page, H, D, Dv, window = "cuda", getattr(torch, dtype), 64, 32, 8, 32, 5
    n = 65600 if single else 262400
    g = torch.Generator(device=dev).manual_seed(3)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev).to(dt)
    q, half = rnd(n, H * D), n // 2
    pages = list(range(n // page))
    k, v = rnd(n, D), rnd(n, Dv)

    def run(lo, hi):
        if single:                                                   # request b attends to the keys of page b % pages
            batch = LO.RaggedBatch.build([1] * (hi - lo), [b % page for b in range(lo, hi)], [0] * (hi - lo), [[b % len(pages)] for b in range(lo, hi)], page, dev)
        else:
            batch = LO.RaggedBatch.build([hi - lo], [lo], [0], [pages], page, dev)
        out = LO.attn_sweep(q[lo:hi].contiguous(), k, v, batch, H, 1, D, Dv, D ** -0.5, window)
        assert any(t.shape[0] > 65535 for key, t in batch._tiles.items() if torch.is_tensor(t)) == (hi - lo == n)
        return out

    assert torch.equal(run(0, n), torch.cat([run(0, half), run(half, n)]))


@pytest.mark.parametrize("built", [False, True])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), float("-inf")])
def test_sinks_that_are_not_finite(monkeypatch, built, value):
    """A sink that is not a number, or infinite, leaves its head's outputs none; one at minus infinity takes nothing; other heads' outputs are what they were, bit for bit.  On built keys a
    wavefront's rows are all of one head, on the pools' of several."""
    from jacobiforcing_amd import layer_ops as LO
    dev, H, G, D, R, rd = "cuda", 16, 4, 64, 128, 32
    g = torch.Generator(device=dev).manual_seed(3)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev).bfloat16()
    counts, starts, pages = [1100, 131], [0, 37], [list(range(18)), list(range(18, 21))]
    batch = LO.RaggedBatch.build(counts, starts, [0, 1], pages, 64, dev)
    q, pool, n = rnd(1231, H * (D + (rd if built else 0))), rnd(21 * 64, R + rd if built else G * D), 1231
    v, uk, uv = rnd(21 * 64, G * D), rnd(H, D, R), rnd(H, R, D)
    monkeypatch.setattr(LO, "_latent_built_requests", lambda *a: [0, 1])

    def run(sink):
        if built:
            return LO.latent_attention(q.clone(), pool, torch.cat([uk.reshape(H * D, R), uv.transpose(1, 2).reshape(H * D, R)]).contiguous(), uk, uv, batch, H, D, R, rd, D, 0, None, None, 0, 0.02, 0, sink=sink)
        out = LO.attn_sweep(q, pool, v, batch, H, G, D, D, 0.125, 0, sink=sink)
        assert ("longest first", 32, None) in batch._tiles, "the 128-row form did not run"
        return out
    sink = torch.randn(H, generator=g, device=dev)
    want, sink[5] = run(sink).view(n, H, D), value
    got = run(sink).view(n, H, D)
    if value == float("-inf"):
        sink[5] = -1e30
        assert torch.equal(got[:, 5], run(sink).view(n, H, D)[:, 5]) and bool(got.isfinite().all())
    else:
        assert bool(got[:, 5].isnan().all())
    got[:, 5] = want[:, 5]
    assert torch.equal(got, want)


# sums of products of small whole numbers, exact in 32 bits, times 2 ** (2 * up): scores of any size that tie or lie apart by one unit of theirs
@pytest.mark.parametrize("up,scale", [(20, 2.0 ** -3), (30, -2.0 ** -3), (50, 2.0 ** -40), (53, 2.0 ** -108), (53, -2.0 ** -108), (53, 0.0), (0, float("nan"))])
def test_scores_and_scales_of_any_size(up, scale):
    from jacobiforcing_amd import layer_ops as LO
    dev, H, G, D = "cuda", 16, 4, 64
    g = torch.Generator(device=dev).manual_seed(4)
    whole = lambda *s: torch.randint(-2, 3, s, generator=g, device=dev).bfloat16() * 2.0 ** up
    counts, starts, pages = [1100, 131], [0, 37], [list(range(18)), list(range(18, 21))]
    q, k, v = whole(1231, H * D), whole(21 * 64, G * D), torch.randn(21 * 64, G * D, generator=g, device=dev).bfloat16()
    batch = LO.RaggedBatch.build(counts, starts, [0, 1], pages, 64, dev)
    got = LO.attn_sweep(q, k, v, batch, H, G, D, D, scale, 0, float_out=True)
    assert ("longest first", 32, None) in batch._tiles, "the 128-row form did not run"
    if scale != scale:
        assert bool(got.isnan().all())
        return
    want = reference(q, k, v, starts, counts, pages, 64, H, G, G, D, D, scale, 0, 0, 0.0, None)
    err = (got.double() - want).abs()      # weights are rounded to bfloat16 once, as in test_wide_tiles
    assert bool(got.isfinite().all()) and err.max() < 2.0 ** -7 * want.abs().max() and err.norm() < 2.0 ** -8 * want.norm()
