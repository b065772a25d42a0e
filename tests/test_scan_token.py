"""The linear recurrence of a decoding step (scan_token_kernel): at the edges of its rows and columns, against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
dev = "cuda"


# depths of one, two and four rows a thread, beside them; columns of one thread, of a workgroup and beside it; a request alone, none with tokens of its own, several tokens beside none; as many heads as it takes, and more, which the wavefronts do
@pytest.mark.parametrize("D", [1, 10, 63, 64, 65, 128, 130, 256])
@pytest.mark.parametrize("H,G,Dv,counts", [(1, 1, 4, [1]), (6, 2, 20, [1, 1, 0, 1]), (8, 8, 16, [1] * 5), (4, 1, 132, [0, 3, 1, 0]), (3, 3, 128, [1, 1]), (128, 1, 4, [1] * 16), (241, 1, 4, [1] * 17)])
@pytest.mark.parametrize("fixed,dtype,act", [(True, torch.bfloat16, False), (False, torch.bfloat16, False), (False, torch.float32, True)])
def test_one_token_each(D, H, G, Dv, counts, fixed, dtype, act):
    from jacobiforcing_amd import layer_ops as LO
    g = torch.Generator(device=dev).manual_seed(D + Dv + H)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    B, N, ld = len(counts), sum(counts), 2 * G * D + H * Dv + 3
    starts, slots = [5 * (b % 2) for b in range(B)], [B - b for b in range(B)]
    batch = LO.RaggedBatch.build(counts, starts, slots, [[b] for b in range(B)], 64, dev)
    src, state = rnd(N, ld).to(dtype), rnd(B + 1, H, D, Dv)
    cols = (3, 3 + G * D, 3 + 2 * G * D)
    kw = dict(decay=torch.rand(H, generator=g, device=dev)) if fixed else dict(dt=rnd(N, H).to(dtype), a_log=0.5 * rnd(H) - 1.0, dt_bias=rnd(H), skip=rnd(H))
    want_state = state.double().clone()
    x = src.double()
    x = x * torch.sigmoid(x) if act else x
    got = LO.linear_scan(src, cols, batch, H, G, D, Dv, state, act=LO.ACT_SILU if act else LO.ACT_NONE, **kw)
    row = 0
    for b, c in enumerate(counts):
        S = want_state[slots[b]]
        A = S.abs() if starts[b] else S * 0                       # the sizes of what is added up
        S = S if starts[b] else S * 0
        for _ in range(c):
            q, k = (x[row, o:o + G * D].view(G, D).repeat_interleave(H // G, 0) for o in cols[:2])
            v = x[row, cols[2]:].view(H, Dv)
            u = torch.ones(H, device=dev, dtype=torch.float64) if fixed else torch.nn.functional.softplus(kw["dt"][row].double() + kw["dt_bias"].double())
            a = kw["decay"].double() if fixed else torch.exp(-kw["a_log"].double().exp() * u)
            new = k[:, :, None] * (u[:, None] * v)[:, None, :]
            S, A = a[:, None, None] * S + new, a[:, None, None] * A + new.abs()
            skip = 0 if fixed else kw["skip"].double()[:, None] * v
            want, size = (S * q[:, :, None]).sum(1) + skip, (A * q[:, :, None].abs()).sum(1) + (0 if fixed else skip.abs())
            # up to four sums in a thread, six exchanges, three more and the skip; an exponential of an argument of a few, silu and softplus to a few 2 ** -24 each
            assert bool(((got[row].view(H, Dv).double() - want).abs() <= 2.0 ** -24 * 64 * size + 1e-30).all())
            row += 1
        if c:
            assert bool(((state[slots[b]].double() - S).abs() <= 2.0 ** -24 * 64 * A + 1e-30).all())
            want_state[slots[b]] = state[slots[b]].double()
    assert torch.equal(state.double(), want_state)                # nobody else's state


# columns beside fours, a state beside 16-byte borders, more tokens than requests, more heads than the form takes
@pytest.mark.parametrize("H,Dv,counts,off", [(2, 18, [1, 1], 0), (2, 16, [1, 1], 1), (2, 16, [2, 1], 0), (2, 16, [1, 3], 0), (3, 20, [4, 0, 2], 0), (1100, 4, [1, 1], 0)])
def test_what_the_wavefronts_keep(H, Dv, counts, off):
    """The same numbers by the form before: every token of every request, and the states that it leaves."""
    from jacobiforcing_amd import layer_ops as LO
    g = torch.Generator(device=dev).manual_seed(H + Dv)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    B, D, starts = len(counts), 12, [3, 0, 7][:len(counts)]
    batch = LO.RaggedBatch.build(counts, starts, list(range(B)), [[b] for b in range(B)], 64, dev)
    src, state = rnd(sum(counts), 2 * H * D + H * Dv), rnd(B * H * D * Dv + off)[off:].view(B, H, D, Dv)
    assert sum(counts) > B or Dv % 4 or state.data_ptr() % 16 or B * H > 2048
    kept, decay = state.double(), torch.rand(H, generator=g, device=dev)
    got, row = LO.linear_scan(src, (0, H * D, 2 * H * D), batch, H, H, D, Dv, state, act=LO.ACT_NONE, decay=decay), 0
    for b, c in enumerate(counts):
        S = kept[b] if starts[b] else kept[b] * 0                  # a request that begins has no state
        A = S.abs()
        for _ in range(c):
            q, k, v = src[row, :H * D].double().view(H, D), src[row, H * D:2 * H * D].double().view(H, D), src[row, 2 * H * D:].double().view(H, Dv)
            new = k[:, :, None] * v[:, None, :]
            S, A = decay.double()[:, None, None] * S + new, decay.double()[:, None, None] * A + new.abs()
            # sums of twelve products and what the tokens before have left, a few 2 ** -24 of their sizes each
            assert bool(((got[row].view(H, Dv).double() - (S * q[:, :, None]).sum(1)).abs() <= 2.0 ** -24 * 64 * (A * q[:, :, None].abs()).sum(1) + 1e-30).all()), (b, row)
            row += 1
        assert bool(((state[b].double() - (S if c else kept[b])).abs() <= 2.0 ** -24 * 64 * A * (c > 0)).all()), b
