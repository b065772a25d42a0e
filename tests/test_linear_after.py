"""Products whose launch makes the rows itself (linear_after_kernel): against the launches that made them before, and 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
dev = "cuda"


def _rnd(seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    return lambda *s: torch.randn(*s, generator=g, device=dev)


def _close(got, want64, w, operand_err):
    """A product of operands off by ``operand_err`` of their size each, rounded to bfloat16: 2 ** -8 of the result and the operands' errors, which the sum averages."""
    assert (got.double() - want64).norm() <= (2.0 ** -8 + operand_err) * want64.norm()


# depths within one pass of the workgroup, two and four, beside whole steps of 64; fewer columns than a tile, columns beside it; the most rows and values
SIZES = [(1, 8, 4), (1, 1024, 1024), (1, 2048, 8192), (3, 2056, 40), (4, 4096, 100), (2, 4104, 16), (1, 8192, 24), (2, 8192, 1000), (4, 72, 17), (4, 520, 2304)]


@pytest.mark.parametrize("n,k,o", SIZES)
@pytest.mark.parametrize("y_type,row,bias", [(torch.bfloat16, False, False), (torch.float32, True, True), (None, True, False), (None, False, True)])
def test_norm(n, k, o, y_type, row, bias):
    from jacobiforcing_amd import layer_ops as LO
    rnd = _rnd(n + k + o)
    x, y, w_post, w_next, add = rnd(n, k), None if y_type is None else (3 * rnd(n, k)).to(y_type), rnd(k), rnd(k), rnd(k) if row else None
    w, b = (rnd(o, k) * k ** -0.5).bfloat16(), rnd(o).bfloat16() if bias else None
    kept = x.clone()
    assert LO._host().norm_linear(x, y, w_post, 1e-5, w_next, add, w, b) is not NotImplemented
    to, out = LO.norm_linear(x, y, w_post, 1e-5, w_next, add, w, b)
    assert torch.equal(x, kept) and to.data_ptr() != x.data_ptr()
    h = LO.sandwich_norm(kept, y, w_post, 1e-5, w_next, torch.bfloat16, add_row=add)
    assert (to - kept).abs().max() <= 2.0 ** -21 * kept.abs().max()                     # the sums of a norm in another order
    _close(out, h.double() @ w.double().T + (0 if b is None else b.double()), w, 2.0 ** -8)      # an operand may round the other way


@pytest.mark.parametrize("n,k,o", SIZES)
@pytest.mark.parametrize("kind,both", [(0, True), (1, True), (2, True), (3, False)])
def test_unit(n, k, o, kind, both):
    from jacobiforcing_amd import layer_ops as LO
    rnd = _rnd(n + k + o + kind)
    z, w, b = rnd(n, 2 * k + 8).bfloat16(), (rnd(o, k) * k ** -0.5).bfloat16(), rnd(o).bfloat16()
    args = (z, 8, k + 8 if both else -1, k, kind)
    assert LO._host().act_linear(*args, 1.5, 1.25, 0.5, w, b) is not NotImplemented
    a = LO.gated_act(*args, 1.5, 1.25, 0.5)
    _close(LO.act_linear(*args, w, b, 1.5, 1.25, 0.5), a.double() @ w.double().T + b.double(), w, 0.0)
    if o <= 4096:
        assert torch.equal(LO.act_linear(*args, w, b, 1.5, 1.25, 0.5), LO.linear(a, w, b))       # the same operand, the same order of sums


@pytest.mark.parametrize("n,k,o", SIZES)
@pytest.mark.parametrize("act,first,scale", [(2, True, 1.0), (4, False, 0.6)])
def test_gated_norm(n, k, o, act, first, scale):
    from jacobiforcing_amd import _native as N, layer_ops as LO
    act = N.JL_ACT_SILU if act == 2 else N.JL_ACT_SIGMOID
    rnd = _rnd(n + k + o + act)
    raw, gate, wn, w = rnd(n, k), rnd(n, k + 24).bfloat16()[:, 8:8 + k], rnd(k), (rnd(o, k) * k ** -0.5).bfloat16()
    assert LO._host().gated_norm_linear(raw, gate, wn, 1e-5, act, first, scale, w, None) is not NotImplemented
    a = LO.gated_norm(raw, gate, wn, 1e-5, act, first, 1, scale)
    _close(LO.gated_norm_linear(raw, gate, wn, 1e-5, act, first, w, 1, scale), a.double() @ w.double().T, w, 2.0 ** -8)


def test_what_the_two_calls_keep():
    """More rows, float weights, autocast, gradients, gates in parts, rows beside 16-byte borders: as before, the residual stream in place."""
    from jacobiforcing_amd import _native as N, layer_ops as LO
    rnd, H = _rnd(5), LO._host()
    x, y, v = rnd(5, 64), rnd(5, 64), rnd(64)
    w = rnd(32, 64).bfloat16()
    assert H.norm_linear(x, y, v, 1e-5, v, None, w, None) is NotImplemented
    to, out = LO.norm_linear(x, y, v, 1e-5, v, None, w)
    assert to is x and out.dtype == torch.bfloat16 and out.shape == (5, 32)
    one = x[:1].contiguous()
    assert H.norm_linear(one, None, None, 1e-5, v, None, w, None) is not NotImplemented
    assert H.norm_linear(one, None, None, 1e-5, v, None, w.float(), None) is NotImplemented and H.norm_linear(one, None, None, 1e-5, v, None, w[:, :56], None) is NotImplemented
    assert LO.norm_linear(one, None, None, 1e-5, v, None, w.float())[1].dtype == torch.float32
    assert H.norm_linear(x.view(-1)[1:65].view(1, 64), None, None, 1e-5, v, None, w, None) is NotImplemented
    with torch.autocast("cuda", dtype=torch.float16):
        assert H.norm_linear(one, None, None, 1e-5, v, None, w, None) is NotImplemented
    leaf = w.clone().requires_grad_()
    assert H.norm_linear(one, None, None, 1e-5, v, None, leaf, None) is NotImplemented
    gate = rnd(1, 64).bfloat16()
    LO.gated_norm_linear(one, gate, v, 1e-5, N.JL_ACT_SILU, True, w, parts=4)
    assert H.gated_norm_linear(one, gate.float(), v, 1e-5, N.JL_ACT_SILU, True, 1.0, w, None) is NotImplemented
    with pytest.raises(ValueError):
        LO.act_linear(gate, 60, -1, 8, LO.ACT_SILU, w[:, :8].contiguous())


@pytest.mark.parametrize("k,o", [(64, 40), (1000, 33), (2048, 4096), (2056, 100), (4096, 1024)])
@pytest.mark.parametrize("n", [2, 3, 4])
def test_rows_are_what_they_are_alone(n, k, o):
    """Rows made at once: each the row of a call of its own, to the last bit."""
    from jacobiforcing_amd import _native as N, layer_ops as LO
    rnd, H = _rnd(n + k + o), LO._host()
    x, y, v, add, gate, z = rnd(n, k), rnd(n, k).bfloat16(), rnd(k), rnd(k), rnd(n, k).bfloat16(), rnd(n, 2 * k).bfloat16()
    w, b = (rnd(o, k) * k ** -0.5).bfloat16(), rnd(o).bfloat16()
    calls = (lambda i: H.norm_linear(x[i], y[i], v, 1e-5, add, add, w, b), lambda i: H.act_linear(z[i], 0, k, k, 1, 1.5, 1.25, 0.5, w, b), lambda i: H.gated_norm_linear(x[i], gate[i], v, 1e-5, N.JL_ACT_SIGMOID, False, 0.7, w, b))
    for call in calls:
        whole = call(slice(0, n))
        assert whole is not NotImplemented
        for r in range(n):
            one = call(slice(r, r + 1))
            for a, c in zip(whole if isinstance(whole, tuple) else (whole,), one if isinstance(one, tuple) else (one,)):
                assert torch.equal(a[r], c[0]), r


def test_where_two_launches_are_the_better_ones():
    """Three rows and more of many columns, or deep ones of more than a few: every workgroup would repeat them."""
    from jacobiforcing_amd import _native as N
    ok = N.layers().jl_linear_after_ok
    for n, k, o in ((1, 8192, 8192), (2, 8192, 8192), (3, 2048, 4096), (4, 2048, 4096), (3, 4096, 1024), (4, 4096, 1024), (4, 8, 4)):
        assert ok(n, k, o) == 1, (n, k, o)
    for n, k, o in ((1, 8200, 64), (2, 8192, 8193), (3, 2048, 4097), (4, 512, 4097), (3, 2056, 1025), (4, 4096, 4096), (3, 4104, 16), (5, 8, 4), (0, 8, 4), (2, 12, 4)):
        assert ok(n, k, o) == 0, (n, k, o)
