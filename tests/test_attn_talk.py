"""Attention with mixed heads in one sweep, at the edges of its tiles (32 keys, 32 or 128 rows), windows and kept tokens, against the same in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,G,D,Dv,window,keep,counts,starts,bias,floats,wgs", [
    (8, 2, 128, 128, 100, 4, [129, 64, 1], [0, 300, 70], "direct", 1 << 28, 512), (4, 4, 64, 32, 0, 0, [200, 33], [5, 0], "lut", 1 << 28, 1), (6, 2, 96, 72, 33, 40, [90, 47, 31], [0, 64, 1000], "direct", 1, 512),
    (16, 1, 8, 8, 64, 70, [50, 20], [150, 0], None, 1 << 28, 64), (12, 4, 40, 128, 1, 3, [40], [7], "lut", 30000, 512), (5, 5, 128, 56, 300, 0, [65, 200], [0, 512], "direct", 1 << 28, 512),
    (8, 2, 128, 128, 1000, 4, [1] * 5, [0, 31, 32, 1500, 999], "direct", 1 << 28, 512), (3, 1, 64, 128, 0, 0, [1, 2, 1], [700, 40, 3], "lut", 1, 512), (16, 8, 24, 16, 50, 2, [3, 1], [64, 10], None, 1 << 28, 1), (32, 1, 16, 24, 40, 1, [1, 2], [90, 33], "lut", 1 << 28, 512), (16, 1, 128, 64, 0, 0, [60, 1], [0, 200], "lut", 1 << 28, 512),
])
def test_talk(monkeypatch, H, G, D, Dv, window, keep, counts, starts, bias, floats, wgs):
    """Portions and single tokens; scratch (``floats``) for all tiles or one at a time, keys whole or shared out (``wgs``); gates per value, strided pools."""
    from jacobiforcing_amd import layer_ops as LO
    dev, page = "cuda", 16
    monkeypatch.setattr(LO, "TALK_SCRATCH_FLOATS", floats)
    monkeypatch.setattr(LO, "TALK_WORKGROUPS", wgs)
    g = torch.Generator(device=dev).manual_seed(H * D + Dv + len(counts))
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    n, B = sum(counts), len(counts)
    need = [-(-(c + s) // page) for c, s in zip(counts, starts)]
    order = torch.randperm(sum(need), generator=torch.Generator().manual_seed(1)).tolist()
    pages = [[order.pop() for _ in range(x)] for x in need]
    batch = LO.RaggedBatch.build(counts, starts, list(range(B)), pages, page, dev)
    kp, vp = rnd(sum(need) * page, G * D + 8).bfloat16()[:, :G * D], rnd(sum(need) * page, G * Dv + 16).bfloat16()[:, 8:8 + G * Dv]
    q, gate, talk = rnd(n, H * D).bfloat16(), rnd(n, H * Dv + 4).bfloat16()[:, 4:], torch.eye(H, device=dev) + 0.4 * rnd(H, H)
    longest = max(c + s for c, s in zip(counts, starts))
    lut = (torch.arange(longest + 50, device=dev).float().sqrt() * 2).int() if bias == "lut" else None
    rel = rnd(int(lut.max()) + 1 if bias == "lut" else 40, H) if bias else None      # direct: distances beyond the table read its last row
    scale = D ** -0.5
    import jacobiforcing_amd._native as N
    assert N.layers().jl_attn_talk_ok(1 if N.JL_BF16 == 1 else N.JL_BF16, H, G, D, Dv, kp.stride(0), vp.stride(0))
    out = LO.attn_window(q, gate, kp, vp, batch, H, G, D, Dv, scale, window, keep, rel, lut, talk, float_out=True)
    rounded = LO.attn_window(q, gate, kp, vp, batch, H, G, D, Dv, scale, window, keep, rel, lut, talk)
    assert torch.equal(rounded, out.bfloat16())
    r0, rep = 0, H // G
    for b, (c, s) in enumerate(zip(counts, starts)):
        tok = torch.tensor([pages[b][j // page] * page + j % page for j in range(c + s)], device=dev)
        k, v = kp[tok].double().view(-1, G, D).repeat_interleave(rep, 1), vp[tok].double().view(-1, G, Dv).repeat_interleave(rep, 1)
        qq = q[r0:r0 + c].double().view(c, H, D)
        sc = (qq.permute(1, 0, 2).contiguous() @ k.permute(1, 2, 0).contiguous()) * scale
        i, j = torch.arange(s, s + c, device=dev).view(-1, 1), torch.arange(c + s, device=dev).view(1, -1)
        if rel is not None:
            d = (i - j).clamp(min=0)
            d = lut[d.clamp(max=lut.numel() - 1)].long() if lut is not None else d.clamp(max=rel.shape[0] - 1)
            sc = sc + rel.double()[d].permute(2, 0, 1)
        see = (j <= i) & (((i - j) < window) | (j < keep) if window > 0 else torch.ones_like(i - j, dtype=torch.bool))
        p = torch.softmax(sc.masked_fill(~see, float("-inf")), -1)
        mixed = torch.einsum("yx,xij->yij", talk.double(), p)
        o = (mixed.contiguous() @ v.permute(1, 0, 2).contiguous()).permute(1, 0, 2) * torch.sigmoid(gate[r0:r0 + c].double().view(c, H, Dv))
        err = (out[r0:r0 + c].double().view(c, H, Dv) - o).norm() / o.norm()
        # scores: float sums of D products times the scale (a few 2 ** -24 of their size, up to about 10); weights to 16 bits of mantissa (2 ** -17), weights and sums cancel by up to 8
        assert err <= 8 * (2.0 ** -17 + 16 * 2.0 ** -24), (b, err.item())
        r0 += c


@pytest.mark.parametrize("H,G,Gv,D,Dv,counts,starts,kw,wgs", [
    (16, 4, 4, 128, 128, [1] * 4, [0, 31, 2000, 999], {}, 2048), (6, 2, 2, 72, 64, [3, 1, 20], [100, 64, 0], dict(window=50, sink=True, gate="head"), 2048),
    (4, 4, 2, 64, 128, [1, 2], [700, 90], dict(chunk=64, float_out=True), 64), (8, 1, 1, 8, 64, [1, 1], [33, 1], dict(softcap=5.0, gate="value", out_scale=0.5), 1),
    (32, 1, 1, 128, 32, [2, 1], [300, 5], dict(sink=True, into=True), 2048), (12, 3, 1, 104, 96, [1] * 3, [63, 64, 500], dict(window=1), 2048),
])
def test_few_tokens(monkeypatch, H, G, Gv, D, Dv, counts, starts, kw, wgs):
    """The form for a few tokens per request without mixed heads: windows, chunks, caps, sinks, gates, shared values, results into wider rows."""
    from jacobiforcing_amd import _native as N
    from jacobiforcing_amd import layer_ops as LO
    dev, page = "cuda", 16
    monkeypatch.setattr(LO, "NARROW_WORKGROUPS", wgs)
    g = torch.Generator(device=dev).manual_seed(H * D + Dv)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    n, B, rep = sum(counts), len(counts), H // G
    need = [-(-(c + s) // page) for c, s in zip(counts, starts)]
    order = torch.randperm(sum(need), generator=torch.Generator().manual_seed(1)).tolist()
    pages = [[order.pop() for _ in range(x)] for x in need]
    batch = LO.RaggedBatch.build(counts, starts, list(range(B)), pages, page, dev)
    kp, vp = rnd(sum(need) * page, G * D + 8).bfloat16()[:, :G * D], rnd(sum(need) * page, Gv * Dv + 16).bfloat16()[:, 8:8 + Gv * Dv]
    q = rnd(n, H * D).bfloat16()
    window, chunk, cap = kw.get("window", 0), kw.get("chunk", 0), kw.get("softcap", 0.0)
    sink = rnd(H) if kw.get("sink") else None
    gate = None if "gate" not in kw else rnd(n, H if kw["gate"] == "head" else H * Dv).bfloat16()
    wider = torch.zeros(n, H * Dv + 12, device=dev, dtype=torch.bfloat16) if kw.get("into") else None
    assert N.layers().jl_attn_narrow_ok(N.JL_BF16, H, G, Gv, D, Dv, kp.stride(0), vp.stride(0))
    calls, real = [], N.layers().jl_attn_narrow
    monkeypatch.setattr(N.layers(), "jl_attn_narrow", lambda *a: calls.append(1) or real(*a), raising=False)
    out = LO.attn_sweep(q, kp, vp, batch, H, G, D, Dv, D ** -0.5, window, value_heads=Gv, float_out=kw.get("float_out", False), sink=sink, gate=gate, gate_per_head=kw.get("gate") == "head",
                        chunk=chunk, softcap=cap, out_scale=kw.get("out_scale", 1.0), out=wider[:, 4:4 + H * Dv] if wider is not None else None)
    assert calls, "the form for a few tokens did not run"
    if wider is not None:
        assert not wider[:, :4].any() and not wider[:, 4 + H * Dv:].any()
    r0 = 0
    for b, (c, s) in enumerate(zip(counts, starts)):
        tok = torch.tensor([pages[b][j // page] * page + j % page for j in range(c + s)], device=dev)
        heads = torch.arange(H, device=dev) // rep
        k, v = kp[tok].double().view(-1, G, D)[:, heads], vp[tok].double().view(-1, Gv, Dv)[:, heads % Gv]
        sc = (q[r0:r0 + c].double().view(c, H, D).permute(1, 0, 2).contiguous() @ k.permute(1, 2, 0).contiguous()) * D ** -0.5
        sc = cap * torch.tanh(sc / cap) if cap else sc
        i, j = torch.arange(s, s + c, device=dev).view(-1, 1), torch.arange(c + s, device=dev).view(1, -1)
        see = (j <= i) & ((i - j) < window if window else (j >= i - i % chunk) if chunk else torch.ones_like(i - j, dtype=torch.bool))
        sc = sc.masked_fill(~see, float("-inf"))
        if sink is not None:
            sc = torch.cat([sc, sink.double().view(H, 1, 1).expand(H, c, 1)], -1)
        o = (torch.softmax(sc, -1)[..., :c + s].contiguous() @ v.permute(1, 0, 2).contiguous()).permute(1, 0, 2) * kw.get("out_scale", 1.0)
        if gate is not None:
            z = torch.sigmoid(gate[r0:r0 + c].double())
            o = o * (z.view(c, H, 1) if kw["gate"] == "head" else z.view(c, H, Dv))
        err = (out[r0:r0 + c].double().reshape(c, H, Dv) - o).norm() / o.norm()
        # weights and results are rounded to bfloat16, 2 ** -9 each; the cap's tanh is a few 1e-7 of the cap off
        assert err <= 2 * 2.0 ** -8, (b, err.item())
        r0 += c


@pytest.mark.parametrize("what", ["lowest", "minus infinity", "not a number"])
@pytest.mark.parametrize("counts,starts,wgs", [([70], [0], 1), ([70], [0], 4096), ([1, 1, 2, 1], [0, 5, 0, 900], 4096), ([1, 1, 2, 1], [0, 5, 0, 900], 1)])
def test_values_at_the_types_ends(monkeypatch, what, counts, starts, wgs):
    """A distance bias of the lowest value or of minus infinity on a query's own key (position 0 sees nothing else), and a cached key that is not a number: as the softmax in 64 bits."""
    from jacobiforcing_amd import layer_ops as LO
    dev, page, H, G, D = "cuda", 16, 4, 2, 64
    monkeypatch.setattr(LO, "TALK_WORKGROUPS", wgs)
    g = torch.Generator(device=dev).manual_seed(3)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    n, need = sum(counts), [-(-(c + s) // page) for c, s in zip(counts, starts)]
    at = [sum(need[:b]) for b in range(len(need))]
    batch = LO.RaggedBatch.build(counts, starts, list(range(len(counts))), [list(range(a, a + x)) for a, x in zip(at, need)], page, dev)
    kp, vp, q, talk, rel = rnd(sum(need) * page, G * D).bfloat16(), rnd(sum(need) * page, G * D).bfloat16(), rnd(n, H * D).bfloat16(), torch.eye(H, device=dev) + 0.3 * rnd(H, H), rnd(1000, H)
    if what == "not a number":
        kp[[a * page + 3 for a in at], :D] = float("nan")            # position 3 of every request, under the first key head
    else:
        rel[0, 1] = torch.finfo(torch.float32).min if what == "lowest" else float("-inf")
    stale = torch.full((1 << 22,), float("inf"), device=dev)         # what an allocation of the call may find in its memory
    del stale
    out, r0 = LO.attn_window(q, None, kp, vp, batch, H, G, D, D, D ** -0.5, 0, 0, rel, None, talk, float_out=True).double().view(n, H, D), 0
    for b, (c, s) in enumerate(zip(counts, starts)):
        tok = torch.arange(at[b] * page, at[b] * page + c + s, device=dev)
        k, v = (x[tok].double().view(-1, G, D).repeat_interleave(H // G, 1).permute(1, 0, 2).contiguous() for x in (kp, vp))
        i, j = torch.arange(s, s + c, device=dev).view(-1, 1), torch.arange(c + s, device=dev).view(1, -1)
        sc = q[r0:r0 + c].double().view(c, H, D).permute(1, 0, 2).contiguous() @ k.transpose(1, 2).contiguous() * D ** -0.5 + rel.double()[(i - j).clamp(min=0)].permute(2, 0, 1)
        p = torch.softmax(sc.masked_fill(j > i, float("-inf")), -1)
        want = (torch.einsum("yx,xij->yij", talk.double(), p).contiguous() @ v).permute(1, 0, 2)
        dead = torch.isnan(want).flatten(1).any(1)                   # rows with a sum that is none: all heads, they are mixed
        assert (what != "lowest" or not bool(dead.any())) and torch.equal(torch.isnan(out[r0:r0 + c]).flatten(1).all(1), dead), (b, dead)
        live = out[r0:r0 + c][~dead]
        # as in test_talk
        assert bool(torch.isfinite(live).all()) and (live - want[~dead]).norm() <= 8 * (2.0 ** -17 + 16 * 2.0 ** -24) * want[~dead].norm(), b
        r0 += c


def test_a_key_that_is_not_a_number_reaches_a_decoded_token():
    """... in the form without mixed heads: alone in its share of the keys it must not drop out."""
    from jacobiforcing_amd import layer_ops as LO
    dev, page, H, G, D = "cuda", 64, 4, 2, 64
    g = torch.Generator(device=dev).manual_seed(3)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev).bfloat16()
    batch = LO.RaggedBatch.build([1, 1], [640, 0], [0, 1], [list(range(11)), [11]], page, dev)
    kp, vp, q = rnd(12 * page, G * D), rnd(12 * page, G * D), rnd(2, H * D)
    kp[640, :D] = kp[11 * page, :D] = float("nan")                   # the last key of one request, the only one of the other
    out = LO.attn_sweep(q, kp, vp, batch, H, G, D, D, D ** -0.5, 0).view(2, G, -1)
    assert bool(torch.isnan(out[:, 0]).all()) and bool(torch.isfinite(out[:, 1]).all())


@pytest.mark.parametrize("mixed", [True, False])
@pytest.mark.parametrize("first", [0, 1, 2, 4])
def test_results_into_rows_that_start_anywhere(monkeypatch, mixed, first):
    """Columns of wider rows: stored four at a time where they start at such borders, otherwise by the forms that store single values."""
    from jacobiforcing_amd import _native as N
    from jacobiforcing_amd import layer_ops as LO
    dev, H, G, D = "cuda", 4, 2, 64
    g = torch.Generator(device=dev).manual_seed(3)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev).bfloat16()
    batch = LO.RaggedBatch.build([1, 3], [100, 60], [0, 1], [[0, 1], [2]], 64, dev)
    kp, vp, q, talk = rnd(192, G * D), rnd(192, G * D), rnd(4, H * D), torch.eye(H, device=dev) + 0.2 * torch.randn(H, H, generator=g, device=dev)
    wider = torch.zeros(4, H * D + 8, dtype=torch.bfloat16, device=dev)
    calls, name = [], "jl_attn_talk" if mixed else "jl_attn_narrow"
    real = getattr(N.layers(), name)
    monkeypatch.setattr(N.layers(), name, lambda *a: calls.append(1) or real(*a), raising=False)
    run = (lambda out: LO.attn_window(q, None, kp, vp, batch, H, G, D, D, D ** -0.5, 0, 0, None, None, talk, out=out)) if mixed else \
        lambda out: LO.attn_sweep(q, kp, vp, batch, H, G, D, D, D ** -0.5, 0, out=out)
    want = run(None)
    run(wider[:, first:first + H * D])
    assert len(calls) == (2 if first % 4 == 0 else 1)
    assert not bool(wider[:, :first].any()) and not bool(wider[:, first + H * D:].any())
    # both forms round weights (to bfloat16, or 16 bits) and results
    assert (wider[:, first:first + H * D].double() - want.double()).abs().max() <= 2 * 2.0 ** -8 * want.double().abs().max()


@pytest.mark.parametrize("H,G,Gv,D,Dv,counts,starts,kw", [
    (8, 2, 2, 128, 128, [1] * 3, [127, 0, 60], {}), (8, 2, 2, 128, 128, [1] * 3, [128, 0, 60], {}), (6, 2, 1, 72, 96, [3, 1, 20], [100, 64, 0], dict(gate="value")),
    (4, 1, 1, 64, 32, [2, 1], [700, 3], dict(window=120, sink=True, gate="head")), (4, 1, 1, 64, 64, [2, 1], [700, 3], dict(window=121)), (32, 1, 1, 40, 64, [5], [0], dict(sink=True, chunk=3, float_out=True)),
])
def test_few_keys_are_not_shared_out(monkeypatch, H, G, Gv, D, Dv, counts, starts, kw):
    """Up to NARROW_WHOLE keys: one launch without a scratch, whose results are those of the shares."""
    from jacobiforcing_amd import _native as N
    from jacobiforcing_amd import layer_ops as LO
    dev = "cuda"
    g = torch.Generator(device=dev).manual_seed(D + Dv)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    n, need = sum(counts), [-(-(c + s) // 16) for c, s in zip(counts, starts)]
    at = [sum(need[:b]) for b in range(len(need))]
    batch = LO.RaggedBatch.build(counts, starts, list(range(len(counts))), [list(range(a, a + x)) for a, x in zip(at, need)], 16, dev)
    kp, vp, q = rnd(sum(need) * 16, G * D).bfloat16(), rnd(sum(need) * 16, Gv * Dv).bfloat16(), rnd(n, H * D).bfloat16()
    gate = None if "gate" not in kw else rnd(n, H if kw["gate"] == "head" else H * Dv).bfloat16()
    sink = rnd(H) if kw.get("sink") else None
    seen, real = [], N.layers().jl_attn_narrow
    monkeypatch.setattr(N.layers(), "jl_attn_narrow", lambda a, st: seen.append((a._obj.splits, a._obj.scratch)) or real(a, st), raising=False)
    run = lambda: LO.attn_sweep(q, kp, vp, batch, H, G, D, Dv, D ** -0.5, kw.get("window", 0), value_heads=Gv, float_out=kw.get("float_out", False), sink=sink, gate=gate,
                                gate_per_head=kw.get("gate") == "head", chunk=kw.get("chunk", 0), out_scale=0.75)
    whole = run()
    monkeypatch.setattr(LO, "NARROW_WHOLE", 0)
    shared = run()
    tq = int(N.layers().jl_attn_talk_tile_rows(H, G, 0))
    reach = min(batch.max_pos, kw["window"] + tq if "window" in kw else kw["chunk"] + tq if "chunk" in kw else batch.max_pos)
    assert (seen[0] == (1, None)) == (reach <= 128) and (seen[1][0] > 1) == (reach > 64)
    # each rounds a row's weights and results to bfloat16 once, after other partial maxima
    assert (whole.double() - shared.double()).norm() <= 2 * 2.0 ** -8 * shared.double().norm()
