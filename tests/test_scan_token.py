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


def test_what_the_wavefronts_keep():
    """Columns beside fours, states and more tokens than requests: the same numbers by the form before."""
    from jacobiforcing_amd import layer_ops as LO
    g = torch.Generator(device=dev).manual_seed(1)
    for Dv, counts in ((18, [1, 1]), (16, [2, 1])):
        batch = LO.RaggedBatch.build(counts, [3, 0], [0, 1], [[0], [1]], 64, dev)
        src, state = torch.randn(sum(counts), 2 * 24 + 2 * Dv, generator=g, device=dev), torch.randn(2, 2, 12, Dv, generator=g, device=dev)
        S, decay = state[0].double(), torch.tensor([0.5, 0.9], device=dev)
        got = LO.linear_scan(src, (0, 24, 48), batch, 2, 2, 12, Dv, state, act=LO.ACT_NONE, decay=decay)
        q, k, v = src[0, :24].double().view(2, 12), src[0, 24:48].double().view(2, 12), src[0, 48:].double().view(2, Dv)
        want = ((decay.double()[:, None, None] * S + k[:, :, None] * v[:, None, :]) * q[:, :, None]).sum(1)
        assert (got[0].view(2, Dv).double() - want).norm() <= 2.0 ** -20 * want.norm()
