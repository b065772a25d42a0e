"""The delta rule of long portions in chunks on the matrix cores, at the edges of its chunks of 64 tokens and tiles of 32 columns, against the recurrence in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("H,G,D,Dv,counts,starts,keys,floats", [
    (4, 2, 128, 128, [200, 64, 1, 40], [0, 30, 5, 2], "random", 1 << 30), (3, 3, 64, 33, [129, 65, 63, 300], [0, 0, 7, 1], "random", 1 << 30), (6, 2, 24, 20, [500, 33], [3, 0], "alike", 1),
    (4, 1, 100, 300, [128, 127, 66], [9, 0, 0], "random", 200000), (1, 1, 4, 1, [32], [1], "alike", 1 << 30), (2, 2, 68, 128, [1000], [0], "alike", 1 << 30), (8, 4, 128, 96, [96], [4], "zero", 40000),
])
def test_chunks(monkeypatch, dtype, H, G, D, Dv, counts, starts, keys, floats):
    """Unequal portions (one token among them), slots of new requests hold NaN; decays of one, ordinary ones, beyond the exponent's range; keys that hardly differ; scratch
    (``floats``) for all heads, some, one key head's."""
    from jacobiforcing_amd import layer_ops as LO
    dev, dt, eps, unit_eps = "cuda", getattr(torch, dtype), 1e-5, 1e-6
    monkeypatch.setattr(LO, "DELTA_SCRATCH_FLOATS", floats)
    monkeypatch.setattr(LO, "DELTA_CHUNKS_FROM", min(max(counts), 64))
    g = torch.Generator(device=dev).manual_seed(D + Dv)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    B, n = len(counts), sum(counts)
    qkv = rnd(n, 2 * G * D + H * Dv + 4 + (-H * Dv) % 4)
    cols = (4, 4 + G * D, 4 + 2 * G * D)
    if keys == "alike":
        qkv[:, cols[1]:cols[1] + G * D] = 1 + 0.01 * qkv[:, cols[1]:cols[1] + G * D]
    if keys == "zero":
        qkv[::3, cols[1]:cols[1] + G * D] = 0
    proj = rnd(n, 2 * H + H * Dv + 3).to(dt)
    pcols = (1, 1 + H, 1 + 2 * H)
    proj[5:9, 1:1 + H] = 300.0                                       # a decay of nothing
    proj[:, 1 + H:1 + 2 * H] += 2.0
    a_log, dt_bias = torch.linspace(-12.0, 6.0, H, device=dev), 0.3 * rnd(H)
    norm_w = 1 + 0.1 * rnd(Dv)
    slots = list(range(1, B + 1))
    state = rnd(B + 2, H, D, Dv)
    for s, sl in zip(starts, slots):
        if s == 0:
            state[sl] = float("nan")
    before = state.clone()
    batch = LO.RaggedBatch.build(counts, starts, slots, [[b * 40 + i for i in range(40)] for b in range(B)], 64, dev)
    run = lambda st: LO.delta_rule(qkv, cols, proj, pcols, a_log, dt_bias, norm_w, batch, H, G, D, Dv, unit_eps, D ** -0.5, eps, st)
    got = run(state)
    assert any(k[0] == "long" for k in batch._tiles if isinstance(k, tuple)), "the form in chunks did not run"
    scan_state = before.clone()
    monkeypatch.setattr(LO, "DELTA_CHUNKS_FROM", 1 << 30)
    scan = run(scan_state)
    x64, p64, r0 = qkv.double(), proj.double(), 0
    for b, (c, s) in enumerate(zip(counts, starts)):
        rows, p = x64[r0:r0 + c], p64[r0:r0 + c]
        unit = lambda x: (x / torch.sqrt((x * x).sum(-1, keepdim=True) + unit_eps)).repeat_interleave(H // G, 1)
        q, k = (unit(rows[:, x:x + G * D].view(c, G, D)) for x in cols[:2])
        v = rows[:, cols[2]:cols[2] + H * Dv].view(c, H, Dv)
        gate = p[:, pcols[2]:pcols[2] + H * Dv].view(c, H, Dv)
        dec = torch.exp(-torch.exp(a_log.double()) * torch.nn.functional.softplus(p[:, pcols[0]:pcols[0] + H] + dt_bias.double()))
        beta = torch.sigmoid(p[:, pcols[1]:pcols[1] + H])
        S = before[slots[b]].double() if s else torch.zeros(H, D, Dv, dtype=torch.float64, device=dev)
        o = []
        for t in range(c):
            S = dec[t].view(H, 1, 1) * S
            u = beta[t].view(H, 1) * (v[t] - (k[t].unsqueeze(-2) @ S).squeeze(-2))
            S = S + k[t].unsqueeze(-1) * u.unsqueeze(-2)
            o.append((q[t].unsqueeze(-2) @ S).squeeze(-2) * D ** -0.5)
        o = torch.stack(o)
        o = o / torch.sqrt((o * o).mean(-1, keepdim=True) + eps) * norm_w.double() * torch.nn.functional.silu(gate)
        # 32-bit sums of products either way: as far off as the token by token form, which may be lucky: 5 roundings.  Where keys hardly differ the corrections of a chunk cancel in
        # the outputs: a rounding of each of up to 64
        slack = 64 * 2.0 ** -24 if keys == "alike" else 5 * 2.0 ** -24
        err = lambda x, want: ((x.double() - want).norm() / want.norm()).item()
        sl = slots[b]
        assert err(state[sl], S) <= 1.5 * err(scan_state[sl], S) + slack, (b, "state")
        assert err(got[r0:r0 + c].view(c, H, Dv), o) <= 1.5 * err(scan[r0:r0 + c].view(c, H, Dv), o) + slack, (b, "outputs")
        r0 += c
    assert torch.equal(state[0], before[0]) and torch.equal(state[B + 1], before[B + 1])


@pytest.mark.parametrize("what,value", [("v", float("nan")), ("v", float("inf")), ("k", float("nan")), ("k", float("-inf")), ("a", float("nan")), ("b", float("nan")), ("q", float("inf"))])
@pytest.mark.parametrize("D,Dv", [(64, 40), (128, 128)])
def test_what_is_not_finite_reaches_later_tokens_only(D, Dv, what, value):
    """... of the heads that read it: what other rows and heads hold is what it is without it, bit for bit."""
    from jacobiforcing_amd import layer_ops as LO
    dev, H, G, n = "cuda", 4, 2, 300
    g = torch.Generator(device=dev).manual_seed(7)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    batch = LO.RaggedBatch.build([n, 70], [0, 9], [0, 1], [[0, 1, 2, 3, 4], [5, 6]], 64, dev)
    cols, pcols = (0, G * D, 2 * G * D), (0, H, 2 * H)
    qkv, proj = rnd(n + 70, 2 * G * D + H * Dv), rnd(n + 70, 2 * H + H * Dv)
    a_log, bias, w, start = rnd(H), rnd(H), 1 + 0.1 * rnd(Dv), rnd(2, H, D, Dv)
    run = lambda st: LO.delta_rule(qkv, cols, proj, pcols, a_log, bias, w, batch, H, G, D, Dv, 1e-6, D ** -0.5, 1e-5, st).view(n + 70, H, Dv)
    for t in (0, 21, 40, 63, 64, 190, n - 1):                        # within blocks of 16, 32 and 64 tokens, at their ends, in the last chunk
        states = [start.clone(), start.clone()]
        want = run(states[0])
        x, at, heads = {"q": (qkv, cols[0] + D + 3, [2, 3]), "k": (qkv, cols[1] + D + 3, [2, 3]), "v": (qkv, cols[2] + 2 * Dv + 3, [2]), "a": (proj, pcols[0] + 2, [2]),
                        "b": (proj, pcols[1] + 2, [2])}[what]
        kept, x[t, at] = x[t, at].clone(), value
        got = run(states[1])
        x[t, at] = kept
        others = [h for h in range(H) if h not in heads]
        assert torch.equal(got[:t], want[:t]) and torch.equal(got[n:], want[n:]) and torch.equal(got[:, others], want[:, others]), t
        assert torch.equal(states[1][1], states[0][1]) and torch.equal(states[1][0, others], states[0][0, others]), t
        last = t + 1 if what == "q" else n
        assert bool(torch.isnan(got[t:last, heads]).any(-1).all()) and torch.equal(got[last:n], want[last:n]), t
        assert all(bool(torch.isfinite(states[1][0, h]).all()) == (what == "q") for h in heads), t


@pytest.mark.parametrize("H,G,D,counts,least", [(16, 16, 64, [777] + [40] * 100 + [1], 64), (8, 2, 128, [300, 63, 5, 1, 1], 2), (8, 2, 128, [300] + [8] * 50 + [1], 16), (16, 16, 64, [100] * 30, 0)])
def test_portions_of_all_kinds(H, G, D, counts, least):
    """Steps whose requests go through chunks, columns and the form for short portions behind each other: as without chunks."""
    from jacobiforcing_amd import layer_ops as LO
    dev, g, n, B = "cuda", torch.Generator(device="cuda").manual_seed(H), sum(counts), len(counts)
    assert LO.delta_chunks_from(counts, H, D) == least
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    qkv, proj, a_log, bias, w, start = rnd(n, 2 * G * D + H * D), rnd(n, 2 * H + H * D), rnd(H), rnd(H), 1 + 0.1 * rnd(D), rnd(B, H, D, D)
    outs, states = [], []
    for chunks in (least, 0):
        batch, st = LO.RaggedBatch.build(counts, [b % 5 for b in range(B)], list(range(B)), [list(range(13 * b, 13 * b + 13)) for b in range(B)], 64, dev), start.clone()
        batch._tiles[("delta", H, D)] = chunks
        outs.append(LO.delta_rule(qkv, (0, G * D, 2 * G * D), proj, (0, H, 2 * H), a_log, bias, w, batch, H, G, D, D, 1e-6, D ** -0.5, 1e-5, st).double())
        states.append(st.double())
        assert any(k[0] == "long" for k in batch._tiles if isinstance(k, tuple)) == (chunks > 0)
    # 32-bit sums in another order, a few roundings of 2 ** -24 each, normed
    assert (outs[0] - outs[1]).norm() <= 1e-5 * outs[1].norm() and (states[0] - states[1]).norm() <= 4e-6 * states[1].norm()


@pytest.mark.parametrize("H,G,D", [(8, 2, 128), (8, 8, 64)])
@pytest.mark.parametrize("lo,hi", [(-3.0, 1.0), (-6.0, -4.0)])
def test_chunks_lose_no_more_bits_than_the_columns(H, G, D, lo, hi):
    """Errors against 64 bits of both forms in float, short and long memories: the state's is no larger, the outputs' (normed, so that errors of a row's size drop out of both) at most a sixth larger."""
    from jacobiforcing_amd import layer_ops as LO
    dev, n, errs = "cuda", 1021, {}
    for seed in range(3):
        g = torch.Generator(device=dev).manual_seed(seed)
        rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
        qkv, proj = torch.nn.functional.silu(rnd(n, 2 * G * D + H * D)), rnd(n, 2 * H + H * D)
        a_log, bias, w, start = lo + (hi - lo) * torch.rand(H, generator=g, device=dev), rnd(H), 1 + 0.1 * rnd(D), 0.1 * rnd(1, H, D, D)
        x, p = qkv.double(), proj.double()
        unit = lambda y: (y / torch.sqrt((y * y).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, 1)
        q, k = (unit(x[:, c:c + G * D].view(n, G, D)) for c in (0, G * D))
        v, dec, beta = x[:, 2 * G * D:].view(n, H, D), torch.exp(-torch.exp(a_log.double()) * torch.nn.functional.softplus(p[:, :H] + bias.double())), torch.sigmoid(p[:, H:2 * H])
        S, o = start[0].double(), []
        for t in range(n):
            S = dec[t].view(H, 1, 1) * S
            S = S + k[t].unsqueeze(-1) * (beta[t].view(H, 1) * (v[t] - (k[t].unsqueeze(-2) @ S).squeeze(-2))).unsqueeze(-2)
            o.append((q[t].unsqueeze(-2) @ S).squeeze(-2) * D ** -0.5)
        o = torch.stack(o)
        o = o / torch.sqrt((o * o).mean(-1, keepdim=True) + 1e-5) * w.double() * torch.nn.functional.silu(p[:, 2 * H:].view(n, H, D))
        for form in (0, 64):
            batch, st = LO.RaggedBatch.build([n], [100], [0], [list(range(18))], 64, dev), start.clone()
            batch._tiles[("delta", H, D)] = form
            got = LO.delta_rule(qkv, (0, G * D, 2 * G * D), proj, (0, H, 2 * H), a_log, bias, w, batch, H, G, D, D, 1e-6, D ** -0.5, 1e-5, st)
            for name, a, b in (("out", got.double().view(n, H, D), o), ("state", st[0].double(), S)):
                errs[name, form] = errs.get((name, form), 0.0) + ((a - b).norm() / b.norm()).item()
    assert errs["state", 64] <= errs["state", 0] and errs["out", 64] <= 7 / 6 * errs["out", 0], errs


@pytest.mark.parametrize("H,G,Dv,ld", [(4100, 1025, 1024, 0), (4, 2, 40, (1 << 26) + 8)])
def test_wide_rows(H, G, Dv, ld):
    """Rows of outputs of which 64 lie beyond what a buffer store reaches (and a chunk's last row far beyond 32 bits of bytes in qkv): as the form in columns."""
    from jacobiforcing_amd import layer_ops as LO
    dev, g, n, D = "cuda", torch.Generator(device="cuda").manual_seed(H), 70, 4
    width = 2 * G * D + H * Dv
    qkv, at = torch.empty(n, max(ld, width), device=dev), max(ld, width) - width
    qkv[:, at:].normal_(generator=g)
    proj = torch.empty(n, 2 * H + H * Dv, device=dev, dtype=torch.bfloat16).normal_(generator=g)
    a_log, bias, w, start = (torch.randn(*s, generator=g, device=dev) for s in ((H,), (H,), (Dv,), (1, H, D, Dv)))
    got = []
    for form in (64, 0):
        batch, st = LO.RaggedBatch.build([n], [5], [0], [[0, 1]], 64, dev), start.clone()
        batch._tiles[("delta", H, D)] = form
        out = LO.delta_rule(qkv, (at, at + G * D, at + 2 * G * D), proj, (0, H, 2 * H), a_log, bias, w, batch, H, G, D, Dv, 1e-6, 0.5, 1e-5, st)
        assert any(k[0] == "long" for k in batch._tiles if isinstance(k, tuple)) == (form > 0)
        got.append((out.view(n, H, Dv), st[0]))
    for h in (0, H // 2, H - 1):
        # 32-bit sums in another order, outputs rounded to 8 bits
        o = [(x[0][:, h].double(), x[1][h].double()) for x in got]
        assert (o[0][0] - o[1][0]).norm() <= 2.0 ** -8 * o[1][0].norm() and (o[0][1] - o[1][1]).norm() <= 4e-6 * o[1][1].norm(), h
    assert bool(got[0][0].isfinite().all()) and bool(got[0][1].isfinite().all())
