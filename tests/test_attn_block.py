"""Attention of draft blocks at the edges of its tiles (64 keys, 128 (head, token) rows, shared-out keys), over cache rows, pages and candidate scratch, against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,T,nkv,G,D,kv,lens,kind,wgs", [
    (3, 32, 2, 4, 128, [512, 63, 0], [32, 7, 32], "rows", 384), (2, 16, 2, 7, 64, [64, 1000], [16, 16], "rows", 1), (5, 5, 1, 3, 72, [0, 1, 130, 64, 200], [5, 0, 3, 5, 1], "cand", 384),
    (1, 64, 2, 8, 128, [777], [64], "rows", 384), (4, 33, 3, 1, 8, [100, 31, 32, 33], [33, 30, 33, 2], "pages", 384), (2, 1, 2, 16, 96, [300, 15], [1, 1], "pages", 1),
    (6, 32, 2, 4, 128, [250] * 6, [32, 32, 20, 1, 32, 9], "cand", 1),
])
def test_block(monkeypatch, R, T, nkv, G, D, kv, lens, kind, wgs):
    from jacobiforcing_amd import layer_ops as LO
    dev = "cuda"
    monkeypatch.setattr(LO, "BLOCK_WORKGROUPS", wgs)
    g = torch.Generator(device=dev).manual_seed(R * T + D)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev).bfloat16()
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)
    q = rnd(R, nkv, G * T, D)
    longest = max(a + b for a, b in zip(kv, lens))
    if kind == "pages":
        page = 16
        cols = -(-longest // page)
        order = torch.randperm(R * cols, generator=torch.Generator().manual_seed(3)).view(R, cols)
        k, v = rnd(R * cols, nkv, page, D), rnd(R * cols, nkv, page, D)
        tables = i32([[int(order[r, c]) if c * page < kv[r] + lens[r] else -1 for c in range(cols)] for r in range(R)])
        out = LO.attn_block(q, T, k, v, i32(kv), i32(lens), longest, tables=tables)
        key = lambda x, r: torch.cat([x[order[r, c]] for c in range(cols)], 1)
    else:
        P = R + 1
        k, v = rnd(P, nkv, longest + 3, D), rnd(P, nkv, longest + 3, D)
        prompt = [(2 * r + 1) % P for r in range(R)]
        cand = [r // 2 if kind == "cand" and r % 2 else -1 for r in range(R)]
        ck, cv = (rnd(R, nkv, T + 4, D), rnd(R, nkv, T + 4, D)) if kind == "cand" else (None, None)
        out = LO.attn_block(q, T, k, v, i32(kv), i32(lens), longest, i32(prompt), None, i32(cand), ck, cv)

        def key(x, r):
            row = x[prompt[r]].clone()
            if cand[r] >= 0:
                row[:, kv[r]:kv[r] + lens[r]] = (ck if x is k else cv)[cand[r], :, :lens[r]]
            return row
    out = out.double().view(R, T, nkv, G, D)
    for r in range(R):
        n = kv[r] + lens[r]
        kk, vv = key(k, r).double()[:, :n], key(v, r).double()[:, :n]
        s = (q[r].double().view(nkv, G * T, D) @ kk.transpose(1, 2).contiguous() * D ** -0.5).view(nkv, G, T, n)
        t, j = torch.arange(T, device=dev).view(T, 1), torch.arange(n, device=dev).view(1, n)
        see = (j < kv[r]) | (j - kv[r] <= t)
        want = torch.softmax(s.masked_fill(~see, float("-inf")), -1).view(nkv, G * T, n) @ vv if n else torch.zeros(nkv, G * T, D, dtype=torch.float64, device=dev)
        want = want.view(nkv, G, T, D).permute(2, 0, 1, 3)
        err = (out[r] - want).abs().max().item()
        # weights and outputs are rounded to bfloat16 (2 ** -9 each of values up to 4 or so), scores keep a few 2 ** -24 of their size
        assert err <= 4 * 2.0 ** -8 * max(1.0, want.abs().max().item() / 4), (r, err)


@pytest.mark.parametrize("plan", [(1, 0), (3, 0), (1, 1), (2, 1), (5, 1)])      # shares of the keys, whether wavefronts take keys in groups
@pytest.mark.parametrize("T,G,D,kv,scale,climb", [
    (32, 2, 128, [0, 31, 32, 33, 95, 96, 97, 127, 128, 129, 640], None, 0.), (21, 3, 64, [5, 107, 108, 235, 236], None, 0.), (65, 1, 8, [0, 63, 700], None, 0.), (7, 18, 72, [300, 1, 511], -0.1, 0.),
    (16, 4, 128, [64, 400], 0., 0.), (32, 2, 128, [900, 64, 33], None, 0.1), (32, 4, 64, [700, 257], None, -0.1),
])
def test_shares_and_groups(monkeypatch, plan, T, G, D, kv, scale, climb):
    """Every form at the borders of tiles (32 and 64 keys, 64 and 128 rows) and of rounds (128 keys); scores that climb from key to key (or fall) pass every greatest one before them by a little."""
    from jacobiforcing_amd import layer_ops as LO
    dev, nkv, R = "cuda", 2, len(kv)
    monkeypatch.setattr(LO, "_block_plan", lambda *a: plan)
    g = torch.Generator(device=dev).manual_seed(T * D)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev).bfloat16()
    longest = max(kv) + T
    q, k, v = rnd(R, nkv, G * T, D), rnd(R, nkv, longest, D), rnd(R, nkv, longest, D)
    if climb:
        q[..., 0], k[..., 0] = 16., (torch.arange(longest, device=dev) * climb).bfloat16() * D ** 0.5 / 16
    lens = [T - r % 2 * (T // 3) for r in range(R)]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)
    out = LO.attn_block(q, T, k, v, i32(kv), i32(lens), longest, i32(list(range(R))), scale=scale).double().view(R, T, nkv, G, D)
    t, f = torch.arange(T, device=dev).view(T, 1), D ** -0.5 if scale is None else scale
    for r in range(R):
        n = kv[r] + lens[r]
        kk, vv, j = k[r].double()[:, :n], v[r].double()[:, :n], torch.arange(n, device=dev).view(1, n)
        s = (q[r].double() @ kk.transpose(1, 2).contiguous() * f).view(nkv, G, T, n)
        p = torch.softmax(s.masked_fill((j >= kv[r]) & (j - kv[r] > t), float("-inf")), -1).view(nkv, G * T, n)
        want, size = (x.view(nkv, G, T, D).permute(2, 0, 1, 3) for x in (p @ vv, p @ vv.abs()))
        # weights are rounded to bfloat16 (half of a last place, 2^-7 of the number at most: 2^-8 of each; their sum is of the unrounded ones), the result once more; a score is off by a few
        # 2^-24 of the greatest sum of its products
        tol = 2.0 ** -8 * size + 2.0 ** -8 * want.abs() + 2.0 ** -18 * size * (1 + float(s.abs().max())) + 2.0 ** -16 * size
        assert bool(((out[r] - want).abs() <= tol).all()), (r, float(((out[r] - want).abs() / tol).max()))


@pytest.mark.parametrize("heads,GT,keys,D,plan", [(8, 128, 544, 128, (2, 1)), (128, 128, 544, 128, (1, 1)), (2, 128, 280, 128, (1, 1)), (2, 224, 544, 64, (1, 1)), (40, 128, 4032, 128, (3, 1)), (128, 64, 4032, 128, (2, 1)),
                                                  (48, 128, 4032, 128, (8, 0)), (96, 128, 4032, 128, (5, 0)), (160, 128, 1532, 128, (3, 0)), (192, 128, 1532, 128, (2, 0)), (192, 128, 544, 128, (1, 0)),
                                                  (256, 128, 2032, 128, (2, 0)), (128, 224, 1032, 64, (1, 0)), (128, 224, 2032, 64, (2, 0)), (1024, 256, 9000, 128, (1, 0)), (0, 0, 544, 128, (1, 1)), (4, 128, -1, 128, (1, 1))])
def test_plan(heads, GT, keys, D, plan):
    """Shares and groups as they were measured the fastest, or nearly; what the launch refuses has a plan too."""
    from jacobiforcing_amd import layer_ops as LO
    assert LO._block_plan(heads, GT, keys, D) == plan


@pytest.mark.parametrize("R,T,candidates", [(1, 1, False), (5, 33, True), (64, 32, True), (3, 200, False)])
def test_slots(R, T, candidates):
    from jacobiforcing_amd import layer_ops as LO
    dev = "cuda"
    g = torch.Generator(device=dev).manual_seed(R)
    i32 = lambda lo, hi, *s: torch.randint(lo, hi, s, generator=g, device=dev, dtype=torch.int32)
    pos, prompt, cand, lens = i32(0, 3000, R * T), i32(0, 60000, R), i32(-2, 4, R), i32(0, T + 1, R)
    main, scratch = LO.block_slots(pos, T, prompt, cand, lens, 70000, T + 3, candidates)       # beyond 32 bits
    t, valid = torch.arange(T, device=dev).view(1, T), torch.arange(T, device=dev).view(1, T) < lens.view(R, 1)
    neg = torch.full((), -1, dtype=torch.int64, device=dev)
    assert torch.equal(main.view(R, T), torch.where(valid & (cand < 0).view(R, 1), prompt.long().view(R, 1) * 70000 + pos.view(R, T), neg))
    assert scratch is None if not candidates else torch.equal(scratch.view(R, T), torch.where(valid & (cand >= 0).view(R, 1), cand.long().view(R, 1) * (T + 3) + t, neg))


def test_operands_in_host_memory_are_refused():
    from jacobiforcing_amd import layer_ops as LO
    dev, R, T, D = "cuda", 2, 4, 64
    q, k, v, ck, cv = (torch.zeros(R, 2, n, D, dtype=torch.bfloat16, device=dev) for n in (3 * T, 32, 32, T, T))
    lens, tables, pos = torch.full((R,), T, dtype=torch.int32, device=dev), torch.zeros(R, 1, dtype=torch.int32, device=dev), torch.zeros(R * T, dtype=torch.int32, device=dev)
    good = dict(k=k, v=v, kv_len=lens, row_len=lens, row_prompt=lens * 0, row_cand=lens * 0, ck=ck, cv=cv)
    for name in good:
        with pytest.raises(ValueError):
            LO.attn_block(q, T, max_keys=32, **{**good, name: good[name].cpu()})
    with pytest.raises(ValueError):
        LO.attn_block(q, T, k, v, lens, lens, 32, tables=tables.cpu())
    rows = [pos, lens, lens, lens]
    for i in range(1, 4):
        args = [x.cpu() if j == i else x for j, x in enumerate(rows)]
        with pytest.raises(ValueError):
            LO.block_slots(args[0], T, *args[1:], 32, T, True)
    assert LO.attn_block(q, T, max_keys=32, **good).shape == (R * T, 6 * D)


@pytest.mark.parametrize("plan", [(1, 0), (3, 0), (1, 1), (2, 1)])
@pytest.mark.parametrize("up,scale", [(20, 2.0 ** -3), (30, -2.0 ** -3), (50, 2.0 ** -40), (53, 2.0 ** -108), (53, -2.0 ** -108), (53, 0.0), (0, float("nan"))])
def test_scores_and_scales_of_any_size(monkeypatch, plan, up, scale):
    """Sums of products of small whole numbers, exact in 32 bits, times 2 ** (2 * up): scores of any size that tie or lie apart by one unit of theirs."""
    from jacobiforcing_amd import layer_ops as LO
    dev, R, T, nkv, G, D, n = "cuda", 2, 32, 2, 2, 64, 400
    monkeypatch.setattr(LO, "_block_plan", lambda *a: plan)
    g = torch.Generator(device=dev).manual_seed(4)
    whole = lambda *s: torch.randint(-2, 3, s, generator=g, device=dev).bfloat16() * 2.0 ** up
    q, k, v = whole(R, nkv, G * T, D), whole(R, nkv, n, D), torch.randn(R, nkv, n, D, generator=g, device=dev).bfloat16()
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)
    got = LO.attn_block(q, T, k, v, i32([n - T] * R), i32([T] * R), n, i32([0, 1]), scale=scale).double().view(R, T, nkv, G, D)
    if scale != scale:
        assert bool(got.isnan().all())
        return
    t, j = torch.arange(T, device=dev).view(T, 1), torch.arange(n, device=dev).view(1, n)
    s = (q.double() @ k.double().transpose(2, 3).contiguous() * scale).view(R, nkv, G, T, n).masked_fill(j - (n - T) > t, float("-inf"))
    want = (torch.softmax(s, -1).view(R, nkv, G * T, n) @ v.double()).view(R, nkv, G, T, D).permute(0, 3, 1, 2, 4)
    err = (got - want).abs()               # weights and outputs are rounded to bfloat16, as in test_block
    assert bool(got.isfinite().all()) and float(err.max()) <= 4 * 2.0 ** -8 * max(1.0, float(want.abs().max()) / 4)
