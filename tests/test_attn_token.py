"""Attention of a few tokens whose wavefronts have keys of their own (jl_attn_token.hip): latents, mixed heads and grouped heads at the edges of rows, tiles and shares, against the same in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _step(counts, starts, page):
    from jacobiforcing_amd import layer_ops as LO
    need = [-(-(c + s) // page) for c, s in zip(counts, starts)]
    order = torch.randperm(sum(need), generator=torch.Generator().manual_seed(1)).tolist()
    pages = [[order.pop() for _ in range(x)] for x in need]
    return LO.RaggedBatch.build(counts, starts, list(range(len(counts))), pages, page, "cuda"), pages, sum(need) * page


def _exact(q, k, v, scale, see, sink=None, add=None):
    """[c, H, D], [K, H, D], [K, H, Dv] in 64 bits -> weights [H, c, K] without the sink's, values [H, K, Dv]."""
    sc = q.permute(1, 0, 2).contiguous() @ k.permute(1, 2, 0).contiguous() * scale
    sc = (sc if add is None else sc + add).masked_fill(~see, float("-inf"))
    if sink is not None:
        sc = torch.cat([sc, sink.double().view(-1, 1, 1).expand(-1, sc.shape[1], 1)], -1)
    return torch.softmax(sc, -1)[..., :k.shape[0]].contiguous(), v.permute(1, 0, 2).contiguous()


@pytest.mark.parametrize("H,R,rd,counts,starts,page,window,sink", [
    (16, 512, 64, [1] * 3, [0, 15, 2040], 64, 0, False), (16, 512, 8, [3, 1], [300, 16], 48, 100, True), (5, 384, 64, [2, 1, 3], [700, 127, 0], 16, 0, False), (12, 256, 64, [2, 2], [97, 1000], 64, 0, True),
    (32, 256, 0, [1, 1], [128, 129], 64, 50, False), (8, 128, 32, [4, 9, 1], [31, 513, 1500], 64, 1024, False), (3, 160, 24, [5, 1], [260, 33], 10, 0, False), (16, 32, 8, [2], [33], 64, 17, True),
    (8, 128, 64, [1] * 300, [3] * 300, 4, 0, False), (1, 64, 64, [1], [9000], 64, 0, False),
])
def test_latents(H, R, rd, counts, starts, page, window, sink):
    from jacobiforcing_amd import layer_ops as LO
    g = torch.Generator(device="cuda").manual_seed(H * R + rd)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    batch, pages, tokens = _step(counts, starts, page)
    n, W = sum(counts), R + rd
    pool, q, gate = rnd(tokens, W + 8).bfloat16()[:, :W], rnd(n, H * W).bfloat16(), rnd(n, H).bfloat16()
    sinks = rnd(H) if sink else None
    out, r0 = LO.attn_sweep(q, pool, pool[:, :R], batch, H, 1, W, R, W ** -0.5, window, sink=sinks, gate=gate, gate_per_head=True), 0
    for b, (c, s) in enumerate(zip(counts, starts)):
        if b < 3 or b == len(counts) - 1:
            tok = torch.tensor([pages[b][j // page] * page + j % page for j in range(c + s)], device="cuda")
            k = pool[tok].double()[:, None].expand(-1, H, -1)
            i, j = torch.arange(s, s + c, device="cuda").view(-1, 1), torch.arange(c + s, device="cuda").view(1, -1)
            p, v = _exact(q[r0:r0 + c].double().view(c, H, W), k, k[..., :R], W ** -0.5, (j <= i) & ((i - j < window) | (window == 0)), sinks)
            want = (p @ v).permute(1, 0, 2) * torch.sigmoid(gate[r0:r0 + c].double()).unsqueeze(-1)
            # weights and results are rounded to bfloat16, 2 ** -9 each
            assert (out[r0:r0 + c].double().view(c, H, R) - want).norm() <= 2 * 2.0 ** -8 * want.norm(), b
        r0 += c


@pytest.mark.parametrize("H,G,D,Dv,counts,starts,page,window,keep,bias,wgs", [
    (16, 4, 128, 128, [1] * 3, [0, 16, 2040], 64, 1024, 4, "lut", 256), (16, 1, 128, 128, [1] * 2, [31, 32], 48, 0, 0, "direct", 256), (8, 2, 128, 128, [2, 1], [1500, 77], 64, 100, 40, "lut", 256),
    (8, 4, 64, 64, [1, 2], [640, 0], 16, 0, 0, None, 1), (2, 2, 72, 40, [8, 3], [129, 5], 64, 33, 17, "direct", 256), (1, 1, 8, 8, [16], [300], 10, 16, 3, "direct", 4), (12, 2, 96, 96, [1], [9000], 64, 0, 0, "lut", 256),
])
def test_mixed_heads(monkeypatch, H, G, D, Dv, counts, starts, page, window, keep, bias, wgs):
    from jacobiforcing_amd import layer_ops as LO
    monkeypatch.setattr(LO, "NARROW_WORKGROUPS", wgs)
    g = torch.Generator(device="cuda").manual_seed(H * D + Dv)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    batch, pages, tokens = _step(counts, starts, page)
    n, longest, rep = sum(counts), max(c + s for c, s in zip(counts, starts)), H // G
    assert LO._few(batch, H, 16, 32 * G // H) == max(counts)
    kp, vp, q, gate = rnd(tokens, G * D + 8).bfloat16()[:, :G * D], rnd(tokens, G * Dv).bfloat16(), rnd(n, H * D).bfloat16(), rnd(n, H * Dv).bfloat16()
    talk, lut = torch.eye(H, device="cuda") + 0.4 * rnd(H, H), (torch.arange(longest, device="cuda").float().sqrt() * 2).int() if bias == "lut" else None
    rel = rnd(int(lut.max()) + 1 if bias == "lut" else 40, H) if bias else None
    out, r0 = LO.attn_window(q, gate, kp, vp, batch, H, G, D, Dv, D ** -0.5, window, keep, rel, lut, talk, float_out=True), 0
    for b, (c, s) in enumerate(zip(counts, starts)):
        tok = torch.tensor([pages[b][j // page] * page + j % page for j in range(c + s)], device="cuda")
        k, v = kp[tok].double().view(-1, G, D).repeat_interleave(rep, 1), vp[tok].double().view(-1, G, Dv).repeat_interleave(rep, 1)
        i, j = torch.arange(s, s + c, device="cuda").view(-1, 1), torch.arange(c + s, device="cuda").view(1, -1)
        add = None
        if rel is not None:
            d = (i - j).clamp(min=0)
            add = rel.double()[lut[d].long() if lut is not None else d.clamp(max=rel.shape[0] - 1)].permute(2, 0, 1)
        p, v = _exact(q[r0:r0 + c].double().view(c, H, D), k, v, D ** -0.5, (j <= i) & ((i - j < window) | (j < keep) | (window == 0)), add=add)
        want = (torch.einsum("yx,xij->yij", talk.double(), p).contiguous() @ v).permute(1, 0, 2) * torch.sigmoid(gate[r0:r0 + c].double().view(c, H, Dv))
        # float scores, weights to 16 bits of mantissa (2 ** -17), weights and sums cancel by up to 8
        assert (out[r0:r0 + c].double().view(c, H, Dv) - want).norm() <= 8 * (2.0 ** -17 + 16 * 2.0 ** -24) * want.norm(), b
        r0 += c


def test_a_request_without_tokens_beside_others():
    from jacobiforcing_amd import layer_ops as LO
    g = torch.Generator(device="cuda").manual_seed(5)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    pages, H, G, D = [[0, 1, 2], [3], [4, 5]], 8, 2, 64
    kp, vp, q, pool, ql = rnd(6 * 64, G * D), rnd(6 * 64, G * D), rnd(3, H * D), rnd(6 * 64, 160), rnd(3, H * 160)
    step = LO.RaggedBatch.build([1, 0, 2], [150, 0, 70], [0, 1, 2], pages, 64, "cuda")
    alone = LO.RaggedBatch.build([1, 2], [150, 70], [0, 1], [pages[0], pages[2]], 64, "cuda")
    for run in (lambda b: LO.attn_sweep(q, kp, vp, b, H, G, D, D, 0.1, 0), lambda b: LO.attn_sweep(ql, pool, pool[:, :128], b, H, 1, 160, 128, 0.1, 0)):
        a, b = run(step).double(), run(alone).double()
        assert (a - b).norm() <= 2 * 2.0 ** -8 * b.norm()            # tiles of as many queries, other shares of the keys


@pytest.mark.parametrize("counts,starts", [([1, 2, 1], [5, 40, 900]), ([70], [0])])
@pytest.mark.parametrize("H,G,D", [(8, 2, 128), (4, 4, 64), (8, 4, 96), (6, 1, 40)])
@pytest.mark.parametrize("head", [0, -1])
def test_mixed_heads_with_a_key_that_one_head_never_takes(counts, starts, H, G, D, head):
    """A key whose scores are minus infinity under one key head weighs nothing there and is any other key under the others, in this form as in that of long portions."""
    from jacobiforcing_amd import layer_ops as LO
    g = torch.Generator(device="cuda").manual_seed(H * D + G)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    batch, pages, tokens = _step(counts, starts, 16)
    n, rep, c0 = sum(counts), H // G, head % G
    kp, vp, q, talk = rnd(tokens, G * D).bfloat16(), rnd(tokens, G * D).bfloat16(), rnd(n, H * D).bfloat16(), torch.eye(H, device="cuda") + 0.3 * rnd(H, H)
    q.view(n, H, D)[:, c0 * rep:(c0 + 1) * rep, 2] = q.view(n, H, D)[:, c0 * rep:(c0 + 1) * rep, 2].abs() + 0.5
    for own in pages:
        kp[own[0] * 16 + 3, c0 * D + 2] = float("-inf")
    out, r0 = LO.attn_window(q, None, kp, vp, batch, H, G, D, D, D ** -0.5, 0, 0, None, None, talk, float_out=True), 0
    for b, (c, s) in enumerate(zip(counts, starts)):
        tok = torch.tensor([pages[b][j // 16] * 16 + j % 16 for j in range(c + s)], device="cuda")
        k, v = kp[tok].double().view(-1, G, D).repeat_interleave(rep, 1), vp[tok].double().view(-1, G, D).repeat_interleave(rep, 1)
        i, j = torch.arange(s, s + c, device="cuda").view(-1, 1), torch.arange(c + s, device="cuda").view(1, -1)
        p, v = _exact(q[r0:r0 + c].double().view(c, H, D), k, v, D ** -0.5, j <= i)
        want = (torch.einsum("yx,xij->yij", talk.double(), p).contiguous() @ v).permute(1, 0, 2)
        got = out[r0:r0 + c].double().view(c, H, D)
        # as in test_mixed_heads
        assert bool(want.isfinite().all()) and (got - want).norm() <= 8 * (2.0 ** -17 + 16 * 2.0 ** -24) * want.norm(), b
        r0 += c


@pytest.mark.parametrize("what", ["scores", "scale", "sink"])
@pytest.mark.parametrize("H,R,grouped", [(8, 128, False), (4, 512, False), (6, 64, True)])
@pytest.mark.parametrize("counts,starts", [([2, 1], [9, 40]), ([1, 1], [1000, 700])])
def test_scores_scales_and_sinks_to_the_end_of_the_floats(what, H, R, grouped, counts, starts):
    """Finite scores, scales and sinks of the largest binade, which tie or lie so far apart that only the largest weigh anything: keys whole and shared out."""
    from jacobiforcing_amd import layer_ops as LO
    g = torch.Generator(device="cuda").manual_seed(R)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    batch, pages, tokens = _step(counts, starts, 64)
    n, up, scale = sum(counts), *((-60, 3e38) if what == "scale" else (63, 1.0))
    k, q, sinks = rnd(tokens, R).bfloat16(), torch.zeros(n, H * R, device="cuda").bfloat16(), torch.full((H,), 3e38, device="cuda") if what == "sink" else None
    v = rnd(tokens, R).bfloat16() if grouped else k
    q.view(n, H, R)[..., 0] = 2.0 ** up
    k[:, 0] = torch.tensor([1.0, 1.25, 1.5, 1.75], device="cuda")[torch.arange(tokens, device="cuda") % 4] * 2.0 ** (up if what == "scale" else 64)      # the sink lies between the last two
    out, r0 = LO.attn_sweep(q, k, v if grouped else k[:, :R], batch, H, 1, R, R, scale, 0, sink=sinks, float_out=True), 0
    for b, (c, s) in enumerate(zip(counts, starts)):
        tok = torch.tensor([pages[b][j // 64] * 64 + j % 64 for j in range(c + s)], device="cuda")
        kk, vv = (x[tok].double()[:, None].expand(-1, H, -1) for x in (k, v))
        i, j = torch.arange(s, s + c, device="cuda").view(-1, 1), torch.arange(c + s, device="cuda").view(1, -1)
        p, vv = _exact(q[r0:r0 + c].double().view(c, H, R), kk, vv, float(torch.tensor(scale)), j <= i, sinks)
        want, got = (p @ vv).permute(1, 0, 2)[..., 1:], out[r0:r0 + c].double().view(c, H, R)[..., 1:]
        # weights are rounded to bfloat16; scores of a scale of 3e38 lie around 300, a few 2 ** -24 of which move a weight by less
        assert bool(got.isfinite().all()) and (got - want).norm() <= 2 * 2.0 ** -8 * want.norm(), b
        r0 += c


@pytest.mark.parametrize("H,R,rd,pad,counts,starts,splits", [
    (40, 128, 64, 0, [1, 2], [700, 130], True), (8, 128, 96, 0, [3, 1], [500, 64], True), (4, 256, 64, 4, [1, 1], [900, 31], True), (33, 256, 0, 0, [2], [40], False), (20, 384, 64, 0, [1, 1], [600, 5], True),
    (32, 512, 64, 0, [1] * 2, [1000, 31], True), (16, 512, 128, 0, [2, 1], [300, 17], True), (8, 128, 64, 4, [40, 3], [100, 0], True),
])
def test_latents_that_stay_with_four_wavefronts(monkeypatch, H, R, rd, pad, counts, starts, splits):
    """More heads, wider rotary columns and rows beside 16-byte borders: attn_sweep_kernel, its keys whole and shared out."""
    from jacobiforcing_amd import layer_ops as LO
    g = torch.Generator(device="cuda").manual_seed(H * R + rd)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    batch, pages, tokens = _step(counts, starts, 64)
    n, W, launched, args = sum(counts), R + rd, [], LO._attn_args
    monkeypatch.setattr(LO, "_attn_args", lambda *a: launched.append(args(*a)) or launched[-1])
    pool, q, sinks = rnd(tokens, W + pad).bfloat16()[:, :W], rnd(n, H * W).bfloat16(), rnd(H)
    out, r0 = LO.attn_sweep(q, pool, pool[:, :R], batch, H, 1, W, R, W ** -0.5, 0, sink=sinks), 0
    assert len(launched) == 1 and launched[0].longest == 0 and (launched[0].splits > 1) == splits
    for b, (c, s) in enumerate(zip(counts, starts)):
        tok = torch.tensor([pages[b][j // 64] * 64 + j % 64 for j in range(c + s)], device="cuda")
        k = pool[tok].double()[:, None].expand(-1, H, -1)
        i, j = torch.arange(s, s + c, device="cuda").view(-1, 1), torch.arange(c + s, device="cuda").view(1, -1)
        p, v = _exact(q[r0:r0 + c].double().view(c, H, W), k, k[..., :R], W ** -0.5, j <= i, sinks)
        want = (p @ v).permute(1, 0, 2)
        # weights and results are rounded to bfloat16, 2 ** -9 each
        assert (out[r0:r0 + c].double().view(c, H, R) - want).norm() <= 2 * 2.0 ** -8 * want.norm(), b
        r0 += c


@pytest.mark.parametrize("H,R,counts", [(16, 512, [2, 1]), (8, 512, [4, 3]), (16, 128, [2, 1]), (16, 512, [1, 1])])
def test_latents_in_a_graph(H, R, counts):
    """Portions that the batch's own tables hold in the tiles of one form: a graph of a step that nothing has run before takes that form, and replays it."""
    from jacobiforcing_amd import layer_ops as LO
    g = torch.Generator(device="cuda").manual_seed(R)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    (batch, _, tokens), (again, _, _) = _step(counts, [700, 90], 64), _step(counts, [700, 90], 64)
    W = R + 64
    pool, q = rnd(tokens, W), rnd(sum(counts), H * W)
    run = lambda b: LO.attn_sweep(q, pool, pool[:, :R], b, H, 1, W, R, W ** -0.5, 0)
    want = run(batch).double()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = run(again)
    for _ in range(3):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert (got.double() - want).norm() <= 2 * 2.0 ** -8 * want.norm()      # weights and results are rounded to bfloat16, 2 ** -9 each
