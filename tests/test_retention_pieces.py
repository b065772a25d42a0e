"""Retention of long portions in pieces on the matrix cores, at the edges of its groups of 64 tokens, tiles of 32 and pieces, against the recurrence in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("H,D,Dv,rot,workgroups,counts,starts", [
    (3, 128, 128, 128, 256, [200, 64, 1], [0, 30, 5]), (2, 64, 32, 16, 64, [129, 65, 63, 300], [0, 0, 7, 1]), (4, 20, 100, 0, 8, [1000, 33], [3, 0]),
    (1, 128, 4, 8, 2, [128, 127, 66], [9, 0, 0]), (2, 100, 128, 96, 1, [640], [0]), (1, 4, 68, 0, 256, [32], [1]),
])
def test_pieces(monkeypatch, dtype, H, D, Dv, rot, workgroups, counts, starts):
    """Unequal portions (one token among them), slots of new requests hold NaN; decays of one, nearly none, zero and beyond one."""
    from jacobiforcing_amd import layer_ops as LO
    dev, dt, eps = "cuda", getattr(torch, dtype), 1e-5
    monkeypatch.setattr(LO, "RETENTION_WORKGROUPS", workgroups)
    g = torch.Generator(device=dev).manual_seed(D + Dv)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    B, n = len(counts), sum(counts)
    ld = 2 * H * D + 2 * H * Dv + 12
    cols = (4, 4 + H * D, 4 + 2 * H * D, 4 + 2 * H * D + H * Dv)
    proj = rnd(n, ld).to(dt)
    decay = torch.tensor([0.97, 1.0, 0.0, 1.001][:H] if H > 1 else [1e-30], device=dev)
    slots = list(range(1, B + 1))
    state = rnd(B + 2, H, D, Dv)
    for s, sl in zip(starts, slots):
        if s == 0:
            state[sl] = float("nan")
    before = state.clone()
    a = torch.arange(2048, dtype=torch.float32, device=dev).view(-1, 1) * torch.rand(max(rot, 2) // 2, generator=g, device=dev).view(1, -1)
    cos, sin = (a.cos().contiguous(), a.sin().contiguous()) if rot else (None, None)
    pages = [[b * 40 + i for i in range(40)] for b in range(B)]
    batch = LO.RaggedBatch.build(counts, starts, slots, pages, 64, dev)
    got = LO.retention(proj, cols, batch, H, D, Dv, rot, cos, sin, decay, eps, state)
    assert any(isinstance(k, tuple) and k[0] == "pieces" for k in batch._tiles), "the form in pieces did not run"
    p64, r0 = proj.double(), 0
    for b, (c, s) in enumerate(zip(counts, starts)):
        rows = p64[r0:r0 + c]
        q, k = (rows[:, x:x + H * D].view(c, H, D) for x in cols[:2])
        v, gate = (rows[:, x:x + H * Dv].view(c, H, Dv) for x in cols[2:])
        if rot:
            co, si = cos.double()[s:s + c].unsqueeze(1), sin.double()[s:s + c].unsqueeze(1)
            turn = lambda x: torch.cat([x[..., :rot // 2] * co - x[..., rot // 2:rot] * si, x[..., rot // 2:rot] * co + x[..., :rot // 2] * si, x[..., rot:]], -1)
            q, k = turn(q), turn(k)
        S = before[slots[b]].double() if s else torch.zeros(H, D, Dv, dtype=torch.float64, device=dev)
        o = []
        for t in range(c):
            S = decay.double().view(H, 1, 1) * S + (k[t] * D ** -0.5).unsqueeze(-1) * v[t].unsqueeze(-2)
            o.append((q[t].unsqueeze(-2) @ S).squeeze(-2))
        o = torch.stack(o)
        o = o / torch.sqrt((o * o).mean(-1, keepdim=True) + eps) * torch.nn.functional.silu(gate)
        r = got[r0:r0 + c].double().view(c, H, Dv)
        # sums of up to c * D products of 32 bits; bfloat16 outputs round once more
        assert (state[slots[b]].double() - S).norm() <= 2e-6 * S.norm(), (b, "state")
        assert (r - o).norm() <= (2.0 ** -8 if dtype == "bfloat16" else 5e-6) * o.norm(), (b, "outputs")
        r0 += c
    assert torch.equal(state[0], before[0]) and torch.equal(state[B + 1], before[B + 1])


@pytest.mark.parametrize("dtype,value", [("bfloat16", float("inf")), ("float32", float("nan")), ("float32", float("-inf"))])
def test_values_that_are_not_finite_reach_later_tokens_only(dtype, value):
    """... of their own head and request: what other rows hold is what it is without them, bit for bit."""
    from jacobiforcing_amd import layer_ops as LO
    dev, dt, H, D, Dv = "cuda", getattr(torch, dtype), 3, 64, 96
    g = torch.Generator(device=dev).manual_seed(5)
    counts = [300, 70]
    batch = LO.RaggedBatch.build(counts, [0, 0], [0, 1], [[0, 1, 2, 3, 4], [5, 6]], 64, dev)
    cols = (0, H * D, 2 * H * D, 2 * H * D + H * Dv)
    proj = torch.randn(370, cols[3] + H * Dv, generator=g, device=dev).to(dt)
    run = lambda p, st: LO.retention(p, cols, batch, H, D, Dv, 0, None, None, torch.full((H,), 0.9, device=dev), 1e-5, st).view(370, H, Dv)
    states = [torch.zeros(2, H, D, Dv, device=dev) for _ in range(2)]
    want = run(proj, states[0])
    first = {0: 37, 1: 63, 2: 64}                                    # per head: within a group of 64, its last token, the next one's first
    for h, t in first.items():
        proj[t, cols[2] + h * Dv + 11 * h] = value
    proj[300 + 69, cols[2] + 5] = value                              # the other request's last token
    got = run(proj, states[1])
    for h, t in first.items():
        assert torch.equal(got[:t, h], want[:t, h]) and bool(torch.isnan(got[t:300, h]).any(-1).all()), h
        assert torch.equal(got[300:369, h], want[300:369, h]) and not bool(torch.isfinite(states[1][0, h]).all())
    assert bool(torch.isnan(got[369, 0]).any()) and torch.equal(got[369, 1:], want[369, 1:]) and torch.equal(states[1][1, 1:], states[0][1, 1:])


@pytest.mark.parametrize("H,D,counts,least", [(32, 128, [8] + [1] * 20 + [40, 7], 8), (64, 64, [70, 3, 9, 1, 200], 8), (40, 100, [20, 130] + [1] * 11 + [6], 8), (48, 20, [1] * 50 + [20, 9], 13)])
def test_portions_of_both_kinds(H, D, counts, least):
    """Steps whose short portions go through the scan behind the others' pieces: as all of them through the scan."""
    from jacobiforcing_amd import layer_ops as LO
    dev, g, n, B = "cuda", torch.Generator(device="cuda").manual_seed(H), sum(counts), len(counts)
    assert LO.retention_pieces_from(counts, H, D) == least
    starts = [(7 * b) % 30 for b in range(B)]
    run = lambda batch, st: LO.retention(proj, (0, H * D, 2 * H * D, 3 * H * D), batch, H, D, D, 0, None, None, decay, 1e-5, st)
    proj, decay, start = torch.randn(n, 4 * H * D, generator=g, device=dev), torch.linspace(0.9, 1.0, H, device=dev), torch.randn(B, H, D, D, generator=g, device=dev)
    outs, states = [], []
    for scan in (False, True):
        batch, st = LO.RaggedBatch.build(counts, starts, list(range(B)), [list(range(4 * b, 4 * b + 4)) for b in range(B)], 64, dev), start.clone()
        if scan:
            batch._tiles[("retention", H, D)] = 0
        outs.append(run(batch, st).double())
        states.append(st.double())
        assert any(k[0] == "long" for k in batch._tiles if isinstance(k, tuple)) != scan
    short = torch.repeat_interleave(torch.tensor([c < least for c in counts], device=dev), torch.tensor(counts, device=dev))
    assert torch.equal(outs[0][short], outs[1][short])
    # sums of 32-bit products in another order, normed: as in test_pieces
    assert (outs[0] - outs[1]).norm() <= 1e-5 * outs[1].norm() and (states[0] - states[1]).norm() <= 4e-6 * states[1].norm()


@pytest.mark.parametrize("D,Dv", [(96, 64), (20, 100), (130, 200), (33, 300), (128, 128)])
def test_short_portions_with_infinities(D, Dv):
    """Sums of a column that are infinite (keys and queries of one sign) stay infinite where the kernel's rows are more than D: the other columns of the head come to zero under their norm."""
    from jacobiforcing_amd import layer_ops as LO
    dev, H, counts, starts = "cuda", 2, [3, 1, 5], [0, 4, 2]
    g, n = torch.Generator(device=dev).manual_seed(D), sum(counts)
    cols = (0, H * D, 2 * H * D, 2 * H * D + H * Dv)
    proj = torch.randn(n, cols[3] + H * Dv, generator=g, device=dev)
    proj[:, :cols[2]].abs_()
    start, decay = torch.rand(3, H, D, Dv, generator=g, device=dev), torch.tensor([0.9, 0.5], device=dev)
    proj[1, cols[2] + 7], proj[3, cols[2] + Dv + 9], proj[6, cols[2] + Dv - 1] = float("inf"), float("inf"), float("-inf")
    batch, state = LO.RaggedBatch.build(counts, starts, [0, 1, 2], [[0], [1], [2]], 64, dev), start.clone()
    got = LO.retention(proj, cols, batch, H, D, Dv, 0, None, None, decay, 1e-5, state).view(n, H, Dv)
    assert not any(isinstance(k, tuple) and k[0] in ("pieces", "long") for k in batch._tiles)
    p, r0 = proj.double(), 0
    for b, (c, s) in enumerate(zip(counts, starts)):
        S = start[b].double() if s else torch.zeros(H, D, Dv, dtype=torch.float64, device=dev)
        for t in range(r0, r0 + c):
            q, k = (p[t, x:x + H * D].view(H, D) for x in cols[:2])
            v, gate = (p[t, x:x + H * Dv].view(H, Dv) for x in cols[2:])
            S = decay.double().view(H, 1, 1) * S + (k * D ** -0.5).unsqueeze(-1) * v.unsqueeze(-2)
            o = (q.unsqueeze(-1) * S).sum(-2)
            o = o / torch.sqrt((o * o).mean(-1, keepdim=True) + 1e-5) * torch.nn.functional.silu(gate)
            ok = o.isfinite()
            assert torch.equal(got[t].isfinite(), ok) and torch.allclose(got[t][ok].double(), o[ok], rtol=2e-5, atol=2e-5), (b, t)
        assert torch.equal(state[b].isfinite(), S.isfinite())
        r0 += c


@pytest.mark.parametrize("what,dtype", [(w, d) for w in ("state", "key", "query", "earlier value") for d in ("bfloat16", "float32")] + [("large value", "float32"), ("large query", "float32")])
def test_infinities_and_numbers_beyond_bfloat16(monkeypatch, what, dtype):
    """An infinite state column or key, and floats that lie beyond bfloat16's greatest number, give what the scan gives: sums of one sign stay infinite, finite ones finite, and no token in front is
    reached.  (Values that are not finite spoil their own piece's rows from their token on; those of a later piece see an infinite state.)"""
    from jacobiforcing_amd import layer_ops as LO
    monkeypatch.setattr(LO, "RETENTION_WORKGROUPS", 1024)
    dev, dt, H, D, Dv, counts, starts = "cuda", getattr(torch, dtype), 2, 64, 96, [300, 70], [5, 9]
    g = torch.Generator(device=dev).manual_seed(7)
    cols, rot = (0, H * D, 2 * H * D, 2 * H * D + H * Dv), 0
    proj = torch.randn(370, cols[3] + H * Dv, generator=g, device=dev)
    proj[:, :cols[2]] = proj[:, :cols[2]].abs() * 0.1 + 0.01                                  # queries and keys above zero: an infinity stays one
    start = torch.rand(2, H, D, Dv, generator=g, device=dev) + 0.1
    first, rows = 0, [0, 300]                                                                 # the rows from `first` on of the request are the ones reached
    if what == "state":
        start[0, 1, 3, 40] = float("inf")
    elif what == "key":
        first, proj[150, cols[1] + D + 5] = 150, float("inf")
    elif what == "query":
        first, proj[37, cols[0] + D + 5] = 37, float("inf")
    elif what == "earlier value":
        first, proj[20, cols[2] + Dv + 11] = 64, float("-inf")
    elif what == "large value":
        first, proj[37, cols[2] + Dv + 11] = 37, 3.4e38
        proj[:, :cols[2]] *= 1e-3
    else:
        first, proj[37, cols[0] + D + 5] = 37, 3.4e38
        start *= 1e-30
        proj[:, cols[2]:cols[3]] *= 1e-30
    proj, decay, pages = proj.to(dt), torch.tensor([0.9, 0.97], device=dev), [[0, 1, 2, 3, 4], [5, 6]]
    outs, states = [], []
    for scan in (False, True):
        batch, st = LO.RaggedBatch.build(counts, starts, [0, 1], pages, 64, dev), start.clone()
        if scan:
            batch._tiles[("retention", H, D)] = 0
        outs.append(LO.retention(proj, cols, batch, H, D, Dv, rot, None, None, decay, 1e-5, st).view(370, H, Dv))
        states.append(st)
        assert scan or ("pieces", 64) in batch._tiles
    got, want = outs
    free = torch.ones(370, H, dtype=torch.bool, device=dev)                                   # what nothing reaches
    free[first:300, 1] = False
    assert bool(got[free].isfinite().all()) or what == "earlier value"
    if what == "earlier value":
        free[20:64, 1] = False
        assert bool(got[free].isfinite().all())
    later = torch.zeros_like(free)
    later[first:300, 1] = True
    for a, b in ((got[free], want[free]), (got[later], want[later])):
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.isinf(), b.isinf())
        ok = b.isfinite()
        # sums of 32-bit products in another order, normed; bfloat16 outputs round once more
        assert (a[ok].double() - b[ok].double()).norm() <= (2.0 ** -7 if dtype == "bfloat16" else 1e-5) * max(1.0, float(b[ok].double().norm()))
    a, b = states
    assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.isinf(), b.isinf()) and torch.equal(a[a.isinf()], b[b.isinf()])
    ok = b.isfinite()
    assert (a[ok].double() - b[ok].double()).norm() <= 4e-6 * b[ok].double().norm()
    assert bool(ok.all()) == (what in ("query", "large value", "large query"))


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("D", [64, 128])
def test_states_lean_neither_way(dtype, D):
    """The instructions cut sums towards minus infinity, by 2^-27 of a state's root mean square and more, were it not held with either sign in turn."""
    from jacobiforcing_amd import layer_ops as LO
    dev, H, counts = "cuda", 8, [2048, 1500, 700]
    g = torch.Generator(device=dev).manual_seed(D)
    proj = torch.randn(sum(counts), 4 * H * D, generator=g, device=dev).to(getattr(torch, dtype))
    decay = torch.tensor([1 - 2.0 ** (-5 - 3 * h / H) for h in range(H)], device=dev)
    batch = LO.RaggedBatch.build(counts, [0] * 3, [0, 1, 2], [list(range(32)), list(range(32, 56)), list(range(56, 67))], 64, dev)
    state = torch.zeros(3, H, D, D, device=dev)
    LO.retention(proj, (0, H * D, 2 * H * D, 3 * H * D), batch, H, D, D, 0, None, None, decay, 1e-5, state)
    assert any(isinstance(k, tuple) and k[0] == "pieces" for k in batch._tiles)
    want, r0 = [], 0
    for c in counts:
        k, v = (proj[r0:r0 + c, x * H * D:(x + 1) * H * D].double().view(c, H, D).transpose(0, 1) for x in (1, 2))
        want.append(((k * D ** -0.5 * (decay.double()[:, None] ** torch.arange(c - 1, -1, -1, device=dev))[..., None]).transpose(1, 2).contiguous() @ v.contiguous()))
        r0 += c
    want = torch.stack(want)
    e = (state.double() - want) / want.pow(2).mean().sqrt()
    # a group's cut against its neighbour's is left (measured: 2^-29 to 2^-31), and five times what chance makes of roundings
    assert float(e.mean().abs()) <= 2.0 ** -28.5 + 5 * float(e.std()) / e.numel() ** 0.5, float(e.mean())
