"""Launches of a row (or a few) per workgroup in their forms of four values and of one, and with few and with many rows: widths around the borders of the forms, against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DTYPES = [torch.float32, torch.bfloat16]


def off(t, by):
    """``t`` with its first value ``by`` values behind a border of sixteen bytes."""
    return t.new_empty(t.numel() + by)[by:].view(t.shape).copy_(t)


def close(got, want, size, roundings, dtype):
    """``roundings`` of 2^-24 of ``size``, and the result's own in bfloat16."""
    tol = roundings * 2.0 ** -24 * size + (2.0 ** -8 * want.abs() if dtype == torch.bfloat16 else 0)
    return got.dtype == dtype and bool(((got.double() - want).abs() <= tol + 1e-30).all())


def batch(counts, starts):
    from jacobiforcing_amd import layer_ops as LO
    per = [-(-(c + s) // 8) for c, s in zip(counts, starts)]
    return LO.RaggedBatch.build(counts, starts, list(range(len(counts)))[::-1], [list(range(sum(per[:i]), sum(per[:i + 1]))) for i in range(len(per))], 8, "cuda")


@pytest.mark.parametrize("W,by", [(4, 0), (1020, 0), (1028, 0), (2052, 1), (1022, 0), (4100, 0)])
@pytest.mark.parametrize("dtype", DTYPES)
def test_embedding_and_shift(W, by, dtype):
    from jacobiforcing_amd import layer_ops as LO
    g = torch.Generator(device="cuda").manual_seed(W)
    e, ids = off(torch.randn(9, W, generator=g, device="cuda").to(dtype), by), torch.tensor([8, 0, 3, 3, 7], device="cuda")
    x, c = LO.embed_scale(e, ids, 2.5, True, copy_dtype=torch.bfloat16)
    assert torch.equal(x, e[ids].float() * 2.5) and torch.equal(c, x.bfloat16())
    b = batch([3, 1, 2, 1], [0, 5, 2, 0])
    h, mu, tail = off(torch.randn(7, W, generator=g, device="cuda"), by), torch.rand(W, generator=g, device="cuda"), torch.randn(4, 1, W, generator=g, device="cuda")
    zero = torch.zeros_like(h[0])
    prev = torch.stack([zero, h[0], h[1], tail[2, 0], tail[1, 0], h[4], zero])
    out = LO.token_shift(h, mu, b, tail, dtype)
    assert close(out, h.double() + (prev.double() - h.double()) * mu.double(), h.double().abs() + 2 * (prev.double().abs() + h.double().abs()), 2, dtype)
    assert torch.equal(tail[:, 0], h[[6, 5, 3, 2]])


@pytest.mark.parametrize("Rq,R,rd,by", [(0, 4, 4, 0), (252, 256, 8, 0), (256, 260, 64, 0), (512, 36, 12, 0), (516, 1024, 0, 0), (1028, 512, 64, 0), (2048, 2044, 36, 0), (2052, 512, 64, 0), (768, 512, 64, 1),
                                        (770, 512, 64, 0)])
@pytest.mark.parametrize("pairing", ["JL_ROT_HALVES", "JL_ROT_NEIGHBOURS"])
@pytest.mark.parametrize("dtype", DTYPES)
def test_latents_and_heads(Rq, R, rd, by, pairing, dtype):
    from jacobiforcing_amd import _native as N, layer_ops as LO
    g, n, pairing = torch.Generator(device="cuda").manual_seed(Rq + R), 9, getattr(N, pairing)
    rot = rd if Rq % 8 else rd // 8 * 4                                        # all of the shared key, or its first part
    proj, wq, wk = off(torch.randn(n, Rq + R + rd, generator=g, device="cuda").to(dtype), by), torch.randn(Rq, generator=g, device="cuda").to(dtype), torch.randn(R, generator=g, device="cuda").to(dtype)
    b, ang = batch([n], [5]), torch.randn(64, max(rot // 2, 1), generator=g, device="cuda")
    cos, sin = (ang.cos(), ang.sin()) if rot else (None, None)

    def turned(v):                                                             # [n, heads, rd] in 64 bits, and the size of what is added
        v, half = v.double(), rot // 2
        if not rot:
            return v, v.abs()
        ia = torch.arange(half, device="cuda") * (2 if pairing == N.JL_ROT_NEIGHBOURS else 1)
        ib = ia + (1 if pairing == N.JL_ROT_NEIGHBOURS else half)
        c, s = (t[5:5 + n].double()[:, None] for t in (cos, sin))
        y, size = v.clone(), v.abs()
        y[..., ia], y[..., ib] = v[..., ia] * c - v[..., ib] * s, v[..., ib] * c + v[..., ia] * s
        size[..., ia] = size[..., ib] = v[..., ia].abs() + v[..., ib].abs()
        return y, size

    def normed(v, w):
        v = v.double()
        return v / torch.sqrt((v * v).mean(1, keepdim=True) + 1e-5) * w.double()
    pool = torch.full((16, R + rd), 7.0, dtype=dtype, device="cuda")
    cq = LO.latent_prep(proj, 0, Rq, Rq, R, rd, rot, wq if Rq else None, wk, 1e-5, b, cos, sin, pool, pairing=pairing)
    trips = 32 + max(Rq, R) / 64                                               # roundings of a row's sum, in a row, and of what follows
    if Rq:
        want = normed(proj[:, :Rq], wq)
        assert close(cq, want, want.abs(), trips, dtype)
        alone = LO.latent_prep(proj, 0, Rq, Rq, R, rd, rot, wq, None, 1e-5, b, cos, sin, None, pairing=pairing)
        assert torch.equal(alone, cq)
    want, (key, size) = normed(proj[:, Rq:Rq + R], wk), turned(proj[:, None, Rq + R:])
    rows = pool[b.kv_slot]
    assert close(rows[:, :R], want, want.abs(), trips, dtype) and close(rows[:, R:], key[:, 0], size[:, 0], 3, dtype)
    rest = torch.ones(16, dtype=torch.bool, device="cuda")
    rest[b.kv_slot] = False
    assert bool((pool[rest] == 7.0).all())
    if rot:                                                                    # the heads' rotary parts in place, the rest untouched
        H, D = 3, 12
        q = off(torch.randn(n, H * (D + rd) + 4, generator=g, device="cuda").to(dtype), by)
        before = q.clone()
        N.check_layers(N.layers().jl_rotate_heads(q.data_ptr(), N.JL_BF16 if dtype == torch.bfloat16 else N.JL_F32, n, q.stride(0), H, D, rd, rot, b.pos.data_ptr(), cos.data_ptr(), sin.data_ptr(), 64, pairing,
                                                  torch.cuda.current_stream().cuda_stream))
        parts = lambda t: t[:, :H * (D + rd)].view(n, H, D + rd)
        want, size = turned(parts(before)[..., D:])
        assert close(parts(q)[..., D:], want, size, 3, dtype) and torch.equal(parts(q)[..., :D], parts(before)[..., :D]) and torch.equal(q[:, H * (D + rd):], before[:, H * (D + rd):])


@pytest.mark.parametrize("C,long", [(3072, 1), (3072, 1018), (3072, 1019), (3071, 1021)])
@pytest.mark.parametrize("taps", [2, 4])
@pytest.mark.parametrize("dtype", DTYPES)
def test_short_convolution(C, long, taps, dtype):
    """Requests of one row, of two and of many, from the start and continued, with few and with many rows in the step."""
    from jacobiforcing_amd import layer_ops as LO
    g = torch.Generator(device="cuda").manual_seed(long)
    counts, starts = [1, long, 2, 1, 2], [3, 4, 0, 0, 9]
    b, n = batch(counts, starts), sum(counts)
    x, w = torch.randn(n, C + 4, generator=g, device="cuda").to(dtype), torch.randn(C, taps, generator=g, device="cuda").to(dtype)
    bias, tail = torch.randn(C, generator=g, device="cuda").to(dtype), torch.randn(5, taps - 1, C, generator=g, device="cuda").to(dtype).float()
    want, size, ends, row = [], [], tail.clone(), 0
    for i, (cnt, start) in enumerate(zip(counts, starts)):
        past = tail[4 - i].double() if start else torch.zeros_like(tail[0], dtype=torch.float64)
        seq = torch.cat([past, x[row:row + cnt, 4:].double()])
        parts = torch.stack([seq[j:j + cnt] * w[:, j].double() for j in range(taps)])
        want.append(parts.sum(0) + bias.double())
        size.append(parts.abs().sum(0) + bias.double().abs())
        ends[4 - i], row = seq[-(taps - 1):].float(), row + cnt
    for odt in {torch.float32, dtype}:
        t = tail.clone()
        y = LO.short_conv(x, 4, C, w, b, t, LO.ACT_NONE, bias=bias, out_dtype=odt)
        assert close(y, torch.cat(want), torch.cat(size), taps + 1, odt) and torch.equal(t, ends)
