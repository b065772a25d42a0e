"""The heads' products on both sides of attention over a latent, at the edges of their tiles (32 rows, 32 / 64 / 128 columns, shares of the depth that hold nothing), against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rotated(x, rot, cos, sin, pairing):
    y, half = x.clone(), rot // 2
    for i in range(half):
        u, v = (2 * i, 2 * i + 1) if pairing else (i, i + half)
        y[..., u], y[..., v] = x[..., u] * cos[:, None, i] - x[..., v] * sin[:, None, i], x[..., v] * cos[:, None, i] + x[..., u] * sin[:, None, i]
    return y


@pytest.mark.parametrize("N,H,K,O,rd,rot,pairing,gated", [(1, 3, 8, 8, 0, 0, 0, True), (31, 2, 128, 520, 64, 64, 0, False), (33, 5, 136, 96, 32, 16, 1, False), (64, 1, 256, 64, 0, 0, 0, True),
                                                         (65, 16, 264, 136, 8, 0, 0, False), (32, 4, 512, 128, 0, 0, 0, True), (7, 2, 1032, 40, 16, 16, 1, False), (130, 8, 64, 128, 32, 32, 0, False)])
def test_products(N, H, K, O, rd, rot, pairing, gated):
    from jacobiforcing_amd import layer_ops as LO
    dev = "cuda"
    g = torch.Generator(device=dev).manual_seed(N + K + O)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    head = K + rd + (-(K + rd)) % 8
    wide = rnd(N, H * head + 8).bfloat16()
    x, w, gate = wide[:, 8:], rnd(H, K, O).bfloat16(), rnd(N, H * O + 8).bfloat16()[:, 8:] if gated else None
    cos, sin = (rnd(50, rot // 2) for _ in range(2)) if rot else (None, None)
    batch = LO.RaggedBatch.build([1] * N, [(7 * b) % 50 for b in range(N)], list(range(N)), [[b] for b in range(N)], 64, dev)
    out = LO._host().latent_heads(x, w, head, rd, gate, rot, N, batch.max_pos, batch.pos, cos, sin, pairing)
    assert out is not NotImplemented and out.dtype == torch.bfloat16 and out.shape == (N, H * (O + rd))
    out = out.view(N, H, O + rd).double()
    xs = x.double().view(N, H, head)
    want, size = torch.einsum("nhk,hko->nho", xs[..., :K].cpu(), w.double().cpu()).to(dev), torch.einsum("nhk,hko->nho", xs[..., :K].abs().cpu(), w.double().abs().cpu()).to(dev)
    if gated:
        scale = gate.double().sigmoid().view(N, H, O)
        want, size = want * scale, size * scale
    # float sums of K exact products (and a sigmoid a few units off), then one rounding to bfloat16
    assert bool(((out[..., :O] - want).abs() <= (K + 32) * 2.0 ** -24 * size + 2.0 ** -8 * want.abs()).all())
    if rd:
        p = batch.pos.long()
        turned = _rotated(xs[..., K:K + rd], rot, cos[p].double() if rot else None, sin[p].double() if rot else None, pairing)
        reach = xs[..., K:K + rd].abs().amax(-1, keepdim=True) * 4
        assert bool(((out[..., O:] - turned).abs() <= 2.0 ** -8 * turned.abs() + 2.0 ** -22 * reach).all())


def test_rows_and_heads_that_do_not_meet():
    """A token's values that are not finite reach its own head's outputs and no others."""
    from jacobiforcing_amd import layer_ops as LO
    g = torch.Generator(device="cuda").manual_seed(1)
    x, w = torch.randn(40, 3 * 520, generator=g, device="cuda").bfloat16(), torch.randn(3, 520, 72, generator=g, device="cuda").bfloat16()
    batch = LO.RaggedBatch.build([40], [0], [0], [[0]], 64, "cuda")
    run = lambda v: LO._host().latent_heads(v, w, 520, 0, None, 0, 40, 40, batch.pos, None, None, 0).view(40, 3, 72)
    clean, y = run(x), x.clone()
    y[5, 520 + 519], y[39, 0] = float("inf"), float("nan")
    got = run(y)
    assert not bool(got[5, 1].isfinite().any()) and bool(got[39, 0].isnan().all())
    got[5, 1], got[39, 0] = clean[5, 1], clean[39, 0]
    assert torch.equal(got, clean)


def test_a_part_that_is_not_rotated_needs_no_positions():
    """Through the C interface, where positions and tables may be left out then."""
    import ctypes as C
    from jacobiforcing_amd import _native as N, layer_ops as LO
    g = torch.Generator(device="cuda").manual_seed(6)
    x, w = torch.randn(5, 2 * 48, generator=g, device="cuda").bfloat16(), torch.randn(2, 32, 40, generator=g, device="cuda").bfloat16()
    out = torch.empty(5, 2 * 56, dtype=torch.bfloat16, device="cuda")
    a = N.LatentHeads(x=x.data_ptr(), w=w.data_ptr(), out=out.data_ptr(), N=5, x_ld=96, out_ld=112, H=2, K=32, O=40, x_head=48, out_head=56, rd=16, rot_dims=0, pairing=0)
    N.check_layers(N.layers().jl_latent_heads_run(C.byref(a), LO._stream(x.device)), "jl_latent_heads_run")
    want = x.double().view(5, 2, 48)
    assert torch.equal(out.view(5, 2, 56)[..., 40:], x.view(5, 2, 48)[..., 32:])
    want = (want[..., :32].unsqueeze(-2) @ w.double()).squeeze(-2)
    assert bool(((out.view(5, 2, 56)[..., :40].double() - want).abs() <= 2.0 ** -8 * want.abs() + 64 * 2.0 ** -24 * 32).all())


def test_attention_takes_them_and_agrees(monkeypatch):
    """A layer's result with the package's products and with the library's: the same within their roundings, and nothing is refused or accepted that was not."""
    from jacobiforcing_amd import layer_ops as LO
    dev, H, D, R, rd, Dv = "cuda", 4, 64, 128, 32, 64
    g = torch.Generator(device=dev).manual_seed(2)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    batch = LO.RaggedBatch.build([1, 3, 1], [70, 20, 0], [0, 1, 2], [[0, 1], [2], [3]], 64, dev)
    q, pool = rnd(5, H * (D + rd)).bfloat16(), rnd(256, R + rd).bfloat16()
    uk, uv, cos, sin = (rnd(H, D, R) * D ** -0.5).bfloat16(), (rnd(H, R, Dv) * R ** -0.5).bfloat16(), rnd(80, rd // 2), rnd(80, rd // 2)
    ukv = torch.cat([uk.reshape(H * D, R), uv.transpose(1, 2).reshape(H * Dv, R)]).contiguous()
    for gate, per_head in ((None, False), (rnd(5, H).bfloat16(), True), (rnd(5, H * Dv).bfloat16(), False)):
        run = lambda gate=gate: LO.latent_attention(q.clone(), pool, ukv, uk, uv, batch, H, D, R, rd, Dv, rd, cos, sin, 0, 0.1, 0, gate=gate, gate_per_head=per_head)
        got = run()
        with monkeypatch.context() as m:
            m.setattr(LO, "LATENT_HEADS", 0)
            want = run()
        assert got.shape == want.shape and (got.double() - want.double()).abs().max() <= 3 * 2.0 ** -8 * want.double().abs().max()
    with pytest.raises(ValueError):
        run(rnd(5, H * Dv + 1).bfloat16())


@pytest.mark.parametrize("uk,uv", [((4, 56, 128), (4, 128, 64)), ((4, 8, 128), (4, 128, 64)), ((4, 72, 128), (4, 128, 64)), ((4, 64, 128), (4, 120, 64)), ((4, 64, 128), (4, 136, 64)),
                                   ((4, 64, 120), (4, 128, 64)), ((3, 64, 128), (4, 128, 64))])
def test_up_projections_of_other_sizes_are_refused(uk, uv):
    """Up-projections whose depths are not the heads' are an error, also where they would fit the heads' columns, and whichever products the rule names."""
    from jacobiforcing_amd import layer_ops as LO
    dev, H, D, R, rd, Dv = "cuda", 4, 64, 128, 32, 64
    assert LO.latent_heads(3, H, D, R, Dv, torch.bfloat16)
    batch = LO.RaggedBatch.build([1, 1, 1], [70, 20, 0], [0, 1, 2], [[0, 1], [2], [3]], 64, dev)
    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device=dev)
    cos = torch.zeros(80, rd // 2, device=dev)
    with pytest.raises((RuntimeError, ValueError)):
        LO.latent_attention(z(3, H * (D + rd)), z(256, R + rd), z(H * (D + Dv), R), z(*uk), z(*uv), batch, H, D, R, rd, Dv, rd, cos, cos, 0, 0.1, 0)
