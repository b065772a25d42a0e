"""The residual update and norm, four columns at a time: widths at the edges of its forms, every number of addend rows around four, against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,S,y_dtype,out_dtype,first", [(4, 1, "bfloat16", "bfloat16", False), (252, 3, "float32", "float32", True), (1020, 4, "float32", "bfloat16", False), (1024, 0, "float32", "float32", True),
                                                         (1028, 5, "bfloat16", "bfloat16", True), (2048, 8, "float32", "bfloat16", False), (4100, 2, "bfloat16", "float32", False),
                                                         (8192, 6, "float32", "bfloat16", True), (8196, 4, "float32", "float32", True), (1022, 4, "bfloat16", "bfloat16", True)])
def test_add_rmsnorm(W, S, y_dtype, out_dtype, first):
    from jacobiforcing_amd import layer_ops as LO
    g, N, eps, dt = torch.Generator(device="cuda").manual_seed(W), 5, 1e-5, getattr(torch, out_dtype)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, y, x0, w = rnd(N, W), rnd(N, S, W).to(getattr(torch, y_dtype)) if S else None, rnd(N, W) if first else None, rnd(W).to(dt)
    want = x.double() + (y.double().sum(1) if S else 0) + (x0.double() if first else 0)
    size = x.double().abs() + (y.double().abs().sum(1) if S else 0) + (x0.double().abs() if first else 0)
    normed = want / torch.sqrt((want * want).mean(1, keepdim=True) + eps) * w.double()
    far = x.new_empty(N * W + 1)[1:].view(N, W).copy_(x)                      # rows that do not start at borders of four: one column at a time
    for v in (x, far):
        out = LO.add_rmsnorm(v, y, x0, w, eps, dt)
        assert bool(((v.double() - want).abs() <= (S + 1) * 2.0 ** -24 * size).all())      # one rounding per addend
        # the row's scale is off by its sums' roundings (about W / 1024 + 10 of them in a row), each value by its own, then by the result's
        tol = (S + W / 1024 + 32) * 2.0 ** -24 * (normed.abs() + size / torch.sqrt((want * want).mean(1, keepdim=True)) * w.double().abs()) + (2.0 ** -8 * normed.abs() if dt == torch.bfloat16 else 0)
        assert out.dtype == dt and bool(((out.double() - normed).abs() <= tol).all())
    before = x.clone()
    assert LO.add_rmsnorm(x, None, None, None, eps, None) is None and torch.equal(x, before)
