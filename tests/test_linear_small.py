"""Products of few rows at the edges of their tiles (16 rows of x, 16 / 32 / 64 rows of W, shares of the depth that hold nothing), against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("types", ["bfloat16", "float32", "mixed"])
@pytest.mark.parametrize("N,K,O,bias", [(1, 8, 1, True), (16, 64, 16, False), (17, 72, 15, True), (33, 520, 4096, False), (64, 1024, 4097, True), (31, 1000, 5003, False), (2, 1024, 16400, True),
                                        (1, 4096, 20001, False), (64, 256, 16385, False), (5, 16, 33, True)])
def test_linear(types, N, K, O, bias):
    from jacobiforcing_amd import layer_ops as LO
    dev = "cuda"
    xt, wt = (torch.bfloat16, torch.float32) if types == "mixed" else (getattr(torch, types),) * 2
    assert LO.linear_small(N, K, O, wt.itemsize) or (types != "bfloat16" and N * K > 30000)
    g = torch.Generator(device=dev).manual_seed(N + K + O)
    x = torch.randn(N, K + 16, generator=g, device=dev).to(xt)[:, 8:8 + K]                  # rows apart, 16-byte borders
    w, b = torch.randn(O, K, generator=g, device=dev).to(wt), torch.randn(O, generator=g, device=dev).to(wt) if bias else None
    want = x.double() @ w.double().T + (b.double() if bias else 0)
    size = x.double().abs() @ w.double().abs().T + (b.double().abs() if bias else 0)
    for float_out in (True,) if types == "mixed" else (None, True, False):
        got = LO.linear(x, w, b, float_out)
        assert got.dtype == (torch.float32 if float_out is not None else xt) and got.shape == (N, O)
        # float sums of K exact or once rounded products, in pieces of the depth: at most K / 8 roundings in a row; then one rounding of the result
        tol = (K / 8 + 16) * 2.0 ** -24 * size + (2.0 ** -8 * want.abs() if xt == torch.bfloat16 and not float_out else 0)
        assert bool(((got.double() - want).abs() <= tol).all())
        if float_out is False:
            assert torch.equal(got, got.to(xt).float())


def test_forms_it_does_not_take():
    """Unaligned views, strided columns, no rows, wrong sizes: as the library's product has them."""
    from jacobiforcing_amd import layer_ops as LO
    dev = "cuda"
    w = torch.randn(24, 64, device=dev)
    for x in (torch.randn(3, 65, device=dev)[:, 1:], torch.randn(64, 5, device=dev).t(), torch.randn(0, 64, device=dev), torch.randn(1, 64, device=dev).expand(4, 64)):
        for v in (w, torch.randn(64, 24, device=dev).t()):
            got, want = LO.linear(x, v), x.double() @ v.double().T
            assert got.shape == want.shape and torch.allclose(got.double(), want, atol=1e-4)
    with pytest.raises(RuntimeError):
        LO.linear(torch.randn(3, 60, device=dev), w)
    with pytest.raises(ValueError):
        LO.linear(torch.randn(3, 64, device=dev), w.bfloat16())


@pytest.mark.parametrize("N,K,O,bias", [(65, 8, 1, True), (127, 56, 63, False), (129, 64, 65, True), (1000, 72, 130, False), (64, 1024, 4099, True), (700, 1016, 1000, True), (1, 512, 32000, False), (100, 2048, 8000, True), (513, 1032, 1500, False)])
def test_a_few_hundred_rows(N, K, O, bias):
    from jacobiforcing_amd import layer_ops as LO
    dev, dt = "cuda", torch.bfloat16
    assert LO.linear_mid(N, K, O, dt)
    g = torch.Generator(device=dev).manual_seed(N + K + O)
    x = torch.randn(N, K + 16, generator=g, device=dev).to(dt)[:, 8:8 + K]                  # rows apart, 16-byte borders
    w, b = torch.randn(O, K, generator=g, device=dev).to(dt), torch.randn(O, generator=g, device=dev).to(dt) if bias else None
    want = x.double() @ w.double().T + (b.double() if bias else 0)
    size = x.double().abs() @ w.double().abs().T + (b.double().abs() if bias else 0)
    for float_out in (None, True, False):
        got = LO.linear(x, w, b, float_out)
        assert got.dtype == (torch.float32 if float_out is not None else dt) and got.shape == (N, O)
        # float sums of K exact products: at most K roundings; then one of the result
        tol = (K + 16) * 2.0 ** -24 * size + (2.0 ** -8 * want.abs() if not float_out else 0)
        assert bool(((got.double() - want).abs() <= tol).all())
        if float_out is False:
            assert torch.equal(got, got.to(dt).float())


@pytest.mark.parametrize("dtype", ["bfloat16", "float32", "float16"])
@pytest.mark.parametrize("n", [3, 100])
def test_operands_on_other_devices_and_gradients(dtype, n):
    """Weights or a bias in host memory are refused, types the launches do not know and gradients come from the library, a product over nothing is zero."""
    from jacobiforcing_amd import layer_ops as LO
    dev, dt = "cuda", getattr(torch, dtype)
    x, w, b = torch.randn(n, 64, device=dev).to(dt), torch.randn(32, 64, device=dev).to(dt), torch.randn(32, device=dev).to(dt)
    for args in ((x, w.cpu()), (x, w, b.cpu()), (x, w.cpu(), b)):
        for float_out in (None, True):
            with pytest.raises(RuntimeError):
                LO.linear(*args, float_out=float_out)
    want = x.double() @ w.double().T + b.double()
    assert torch.allclose(LO.linear(x, w, b).double(), want, atol=0.2)
    for i in range(3):
        leaf = [t.clone().requires_grad_(j == i) for j, t in enumerate((x, w, b))]
        LO.linear(*leaf).sum().backward()
        assert leaf[i].grad is not None and bool(leaf[i].grad.any())
    assert torch.equal(LO.linear(x[:, :0].contiguous(), w[:, :0].contiguous()), torch.zeros(n, 32, dtype=dt, device=dev))
