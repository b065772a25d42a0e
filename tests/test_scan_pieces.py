"""The linear recurrence in pieces on the matrix cores: how columns and heads are dealt out to wavefronts (one to four blocks of 32 columns, heads that share q and k in one
workgroup, the last of them incomplete), at the edges of groups of 64 tokens and of widths, against the recurrence in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fixed", [True, False])
@pytest.mark.parametrize("H,G,D,Dv,counts", [
    (3, 3, 128, 128, [64, 1, 200]), (2, 2, 96, 96, [65, 63]), (5, 5, 72, 64, [129, 40]), (9, 1, 128, 64, [130, 33]), (6, 2, 64, 32, [64, 128]), (5, 1, 32, 20, [100, 64, 7]),
    (2, 1, 128, 160, [320]), (1, 1, 4, 4, [191, 2]), (10, 2, 100, 12, [66, 62]),
])
def test_columns_and_heads(monkeypatch, H, G, D, Dv, counts, fixed):
    from jacobiforcing_amd import layer_ops as LO
    monkeypatch.setattr(LO, "SCAN_WAVES", 1)                 # pieces as long as they get: several groups per piece, and ...
    g = torch.Generator(device="cuda").manual_seed(H * 100 + D)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    B, N, starts = len(counts), sum(counts), [0, 3, 0][:len(counts)]
    x = rnd(N, H * Dv + 2 * G * D + 4).bfloat16()
    cols = (H * Dv + G * D + 4, H * Dv, 0)
    kw = dict(decay=torch.rand(H, generator=g, device="cuda")) if fixed else dict(dt=rnd(N, H).bfloat16(), a_log=rnd(H), dt_bias=rnd(H), skip=rnd(H))
    state = rnd(B, H, D, Dv)
    for b, s in enumerate(starts):
        if s == 0:
            state[b] = float("nan")
    pages = [list(range(8 * b, 8 * b + 8)) for b in range(B)]
    for waves in (1, 1 << 20):                               # ... of one group each
        monkeypatch.setattr(LO, "SCAN_WAVES", waves)
        batch, st = LO.RaggedBatch.build(counts, starts, list(range(B)), pages, 64, "cuda"), state.clone()
        got = LO.linear_scan(x, cols, batch, H, G, D, Dv, st, **kw)
        assert any(isinstance(k, tuple) and k[0] == "pieces" for k in batch._tiles), "the form in pieces did not run"
        r0, xd = 0, x.double()
        d = {k: v.double() for k, v in kw.items()}
        for b, (n, s) in enumerate(zip(counts, starts)):
            rows = xd[r0:r0 + n]
            q, k = (rows[:, c:c + G * D].view(n, G, D).repeat_interleave(H // G, 1) for c in cols[:2])
            v = rows[:, :H * Dv].view(n, H, Dv)
            S = state[b].double() if s else torch.zeros(H, D, Dv, dtype=torch.float64, device="cuda")
            for t in range(n):
                u = torch.ones(H, dtype=torch.float64, device="cuda") if fixed else torch.nn.functional.softplus(d["dt"][r0 + t] + d["dt_bias"])
                a = d["decay"] if fixed else torch.exp(-torch.exp(d["a_log"]) * u)
                S = a.view(H, 1, 1) * S + k[t].unsqueeze(2) * (u.view(H, 1) * v[t]).unsqueeze(1)
                o = (S * q[t].unsqueeze(2)).sum(1) + (0 if fixed else d["skip"].view(H, 1) * v[t])
                # 24-bit terms, and weights whose two log decays (up to 2 ** 9 here, rounded to 2 ** -16 each) are off by 2e-5 at most where they are that large
                assert float((got[r0 + t].double().view(H, Dv) - o).norm() / o.norm().clamp_min(1e-3 * D ** 0.5)) < 2e-5, (b, t)
            assert float((st[b].double() - S).norm() / S.norm()) < 2e-5
            r0 += n


@pytest.mark.parametrize("fixed", [True, False])
@pytest.mark.parametrize("H,G,D,Dv,counts", [(3, 3, 128, 128, [64, 1, 200]), (2, 2, 96, 96, [257, 63]), (9, 1, 128, 64, [130, 33]), (5, 1, 32, 20, [100, 440, 7])])
def test_portions_that_stay_whole(monkeypatch, H, G, D, Dv, counts, fixed):
    """One launch, from the slots: as in pieces."""
    from jacobiforcing_amd import layer_ops as LO
    monkeypatch.setattr(LO, "scan_piece_groups", lambda counts, waves: -(-max(counts) // 64))
    test_columns_and_heads(monkeypatch, H, G, D, Dv, counts, fixed)


@pytest.mark.parametrize("op", ["scan", "retention"])
def test_requests_without_tokens(monkeypatch, op):
    """Beside as many pieces as there are requests, all of them one request's: as without the requests that have none, and their states stay."""
    from jacobiforcing_amd import layer_ops as LO
    monkeypatch.setattr(LO, "SCAN_WAVES", 1 << 20)           # pieces of one group each
    monkeypatch.setattr(LO, "RETENTION_WORKGROUPS", 1 << 20)
    g, H, D = torch.Generator(device="cuda").manual_seed(5), 2, 64
    x, start, decay = torch.randn(192, 4 * H * D, generator=g, device="cuda").bfloat16(), torch.randn(3, H, D, D, generator=g, device="cuda"), torch.full((H,), 0.97, device="cuda")
    got = []
    for counts in ([0, 0, 192], [192]):
        b, st = LO.RaggedBatch.build(counts, [0] * len(counts), [0, 1, 2][-len(counts):], [[0, 1, 2]] * len(counts), 64, "cuda"), start.clone()
        if op == "scan":
            o = LO.linear_scan(x, (0, H * D, 2 * H * D), b, H, H, D, D, st, decay=decay)
        else:
            o = LO.retention(x, (0, H * D, 2 * H * D, 3 * H * D), b, H, D, D, 0, None, None, decay, 1e-5, st)
        assert [len(v[0]) for k, v in b._tiles.items() if isinstance(k, tuple) and k[0] == "pieces"] == [3]
        got.append((o, st))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1]) and torch.equal(got[0][1][:2], start[:2])


@pytest.mark.parametrize("pieces", [False, True])
def test_rows_wider_than_the_offsets_of_pieces(monkeypatch, pieces):
    """Rows of outputs whose 64th lies beyond 2 ** 32 bytes, columns beyond a launch's second dimension: in one scan, also where the library is handed pieces."""
    from jacobiforcing_amd import layer_ops as LO
    lib, H, D, Dv, n = LO.N.layers(), 9, 4, (1 << 21) + 64, 40
    g = torch.Generator(device="cuda").manual_seed(9)
    batch = LO.RaggedBatch.build([n], [0], [0], [[0]], 64, "cuda")
    if pieces:
        real, (rec, req) = lib.jl_linear_scan, LO.RaggedBatch.pieces(batch, 64)
        scratch = torch.empty(H * (D * Dv + 1), device="cuda")

        def handed(ap, st):
            a = ap._obj
            a.chunk_rec, a.req, a.scratch, a.chunks = rec.data_ptr(), req.data_ptr(), scratch.data_ptr(), rec.shape[0]
            return real(ap, st)
        monkeypatch.setattr(lib, "jl_linear_scan", handed, raising=False)
    x = torch.empty(n, 2 * D + H * Dv, device="cuda", dtype=torch.bfloat16).normal_(generator=g)
    state, decay = torch.full((1, H, D, Dv), float("nan"), device="cuda"), torch.linspace(0.5, 1.0, H, device="cuda")
    out = LO.linear_scan(x, (0, D, 2 * D), batch, H, 1, D, Dv, state, decay=decay).view(n, H, Dv)
    assert pieces or ("pieces", 64) not in batch._tiles
    q, k, back = x[:, :D].double(), x[:, D:2 * D].double(), torch.arange(n, device="cuda").view(n, 1) - torch.arange(n, device="cuda")
    for h, c in ((0, 0), (4, 1 << 20), (8, Dv - 64)):
        fade = (decay[h].double() ** back.clamp_min(0)).tril()
        v = x[:, 2 * D + h * Dv + c:2 * D + h * Dv + c + 64].double()
        want, S = (q @ k.T * fade) @ v, (k * fade[-1:].T).T @ v
        assert (out[:, h, c:c + 64] - want).norm() <= 2e-6 * want.norm() and (state[0, h, :, c:c + 64] - S).norm() <= 2e-6 * S.norm(), (h, c)


@pytest.mark.parametrize("what,value", [("v", float("nan")), ("v", float("inf")), ("k", float("-inf")), ("q", float("nan")), ("dt", float("nan")), ("dt", float("inf"))])
@pytest.mark.parametrize("H,G,D,Dv", [(6, 2, 64, 40), (4, 4, 128, 128), (5, 1, 20, 20), (2, 2, 96, 64)])
@pytest.mark.parametrize("waves", [1, 1 << 20])
def test_what_is_not_finite_reaches_later_tokens_only(monkeypatch, H, G, D, Dv, waves, what, value):
    """... of the columns and heads that read it, as in the scan token by token; what other rows, columns, heads and requests hold is what it is without it, bit for bit."""
    from jacobiforcing_amd import layer_ops as LO
    monkeypatch.setattr(LO, "SCAN_WAVES", waves)             # pieces of several groups, and of one
    n, per, g = 300, H // G, torch.Generator(device="cuda").manual_seed(H + D)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    batch = LO.RaggedBatch.build([n, 70], [0, 9], [0, 1], [[0, 1, 2, 3, 4], [5, 6]], 64, "cuda")
    cols = (0, G * D, 2 * G * D)
    x, dt, start, kw = rnd(n + 70, 2 * G * D + H * Dv).bfloat16(), rnd(n + 70, H).bfloat16(), rnd(2, H, D, Dv), dict(a_log=rnd(H) - 2, dt_bias=rnd(H), skip=rnd(H), act=LO.ACT_SILU)
    if what != "dt":
        kw = dict(decay=torch.rand(H, generator=g, device="cuda"), skip=kw["skip"])

    def run(pieces):
        st = start.clone()
        monkeypatch.setattr(LO, "SCAN_PIECES_FROM", 32 if pieces else 1 << 30)
        return LO.linear_scan(x, cols, batch, H, G, D, Dv, st, **(kw | (dict(dt=dt) if what == "dt" else {}))).view(n + 70, H, Dv), st
    want, clean = run(True)
    c, h = Dv // 2 + 1, H - 1
    y, at = {"q": (x, cols[0] + (G - 1) * D + 3), "k": (x, cols[1] + (G - 1) * D + 3), "v": (x, cols[2] + h * Dv + c), "dt": (dt, h)}[what]
    for t in (0, 21, 31, 32, 63, 64, 190, n - 1):            # within blocks of 32 and 64 tokens, at their ends, the last
        kept, y[t, at] = y[t, at].clone(), value
        (got, state), (scan, scan_state) = run(True), run(False)
        y[t, at] = kept
        off = torch.zeros(n + 70, H, Dv, dtype=torch.bool, device="cuda")
        off[t:t + 1 if what == "q" else n, h if what in ("v", "dt") else slice(H - per, H), c if what == "v" else slice(0, Dv)] = True
        assert torch.equal(~got.isfinite(), off) and torch.equal(got[~off], want[~off]), t
        assert torch.equal(got.isfinite(), scan.isfinite()) and torch.equal(state.isfinite(), scan_state.isfinite()) and torch.equal(state[state.isfinite()], clean[state.isfinite()]), t


@pytest.mark.parametrize("fixed", [True, False])
@pytest.mark.parametrize("H,G,D,Dv", [(6, 2, 64, 40), (4, 4, 128, 128), (8, 1, 96, 64)])
@pytest.mark.parametrize("whole", [True, False])
def test_operands_keep_their_24_bits(monkeypatch, H, G, D, Dv, fixed, whole):
    """Memories of hundreds of tokens, against 64 bits: a rounding (2 ** -24) of each of the float sums' few halvings and of the operands, 5e-7 at most here; with two bfloat16 terms per operand instead of
    three they would be off by 2 ** -17 each, 8e-6 in the outputs."""
    from jacobiforcing_amd import layer_ops as LO
    monkeypatch.setattr(LO, "scan_piece_groups", lambda counts, waves: -(-max(counts) // 64) if whole else 1)
    g, n = torch.Generator(device="cuda").manual_seed(H * D), 500
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, start = rnd(n, 2 * G * D + H * Dv).bfloat16(), rnd(1, H, D, Dv)
    kw = dict(decay=1 - 2.0 ** -torch.linspace(5, 9, H, device="cuda")) if fixed else dict(dt=rnd(n, H).bfloat16(), a_log=rnd(H) - 5, dt_bias=rnd(H), skip=rnd(H))
    batch, st = LO.RaggedBatch.build([n], [1], [0], [list(range(8))], 64, "cuda"), start.clone()
    got = LO.linear_scan(x, (0, G * D, 2 * G * D), batch, H, G, D, Dv, st, **kw).double().view(n, H, Dv)
    q, k = (x[:, c:c + G * D].double().view(n, G, D).repeat_interleave(H // G, 1) for c in (0, G * D))
    v, S, o = x[:, 2 * G * D:].double().view(n, H, Dv), start[0].double(), []
    d = {key: t.double() for key, t in kw.items()}
    for t in range(n):
        u = torch.ones(H, dtype=torch.float64, device="cuda") if fixed else torch.nn.functional.softplus(d["dt"][t] + d["dt_bias"])
        a = d["decay"] if fixed else torch.exp(-torch.exp(d["a_log"]) * u)
        S = a.view(H, 1, 1) * S + k[t].unsqueeze(2) * (u.view(H, 1) * v[t]).unsqueeze(1)
        o.append((S * q[t].unsqueeze(2)).sum(1) + (0 if fixed else d["skip"].view(H, 1) * v[t]))
    o = torch.stack(o)
    errors = float((got - o).norm() / o.norm()), float((st[0].double() - S).norm() / S.norm())
    assert max(errors) < 1e-6, errors
