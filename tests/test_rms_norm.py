"""Norms of rows in their own type (rms_norm_rows_kernel): at the edges of its vectors, against 64 bits, and what stays the library's."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# one row to beside a workgroup's four, one unit of 16 bytes, widths of 1, 2, 4 and 8 units a lane and beside them
@pytest.mark.parametrize("shape", [(1, 8), (3, 504), (4, 512), (5, 520), (2, 3, 1024), (129, 896), (7, 1032), (9, 2056), (2049, 1024), (3, 4096)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rows(shape, dtype):
    from jacobiforcing_amd import layer_ops as LO
    if dtype == torch.float32 and shape[-1] > 2048:
        shape = shape[:-1] + (2048,)
    g = torch.Generator(device="cuda").manual_seed(shape[-1])
    x, w = (30 * torch.randn(*shape, generator=g, device="cuda")).to(dtype), torch.randn(shape[-1], generator=g, device="cuda").to(dtype)
    x.view(-1, shape[-1])[-1] *= 0
    assert LO._host().rms_norm(x, w, 1e-6) is not NotImplemented
    got, d = LO.rms_norm(x, w, 1e-6), x.double()
    want = d / (d.pow(2).mean(-1, keepdim=True) + 1e-6).sqrt() * w.double()
    assert got.dtype == dtype and got.shape == x.shape
    # float: the sum of W squares, the root and two products; bfloat16: rounded once
    tol = 2.0 ** -21 if dtype == torch.float32 else 2.0 ** -8
    assert bool(((got.double() - want).abs() <= tol * want.abs() + 1e-30).all())


def test_what_the_library_keeps():
    from jacobiforcing_amd import layer_ops as LO
    x, w, H = torch.randn(4, 64, device="cuda"), torch.randn(64, device="cuda"), LO._host()
    assert H.rms_norm(x, w, 1e-6) is not NotImplemented
    for a, b in ((x.half(), w.half()), (x, w.bfloat16()), (x.t().contiguous().t(), w), (x[:, :63].contiguous(), w[:63]), (x.view(-1)[1:65].view(1, 64), w), (x[:0], w), (torch.randn(1, 8192, device="cuda"), torch.randn(8192, device="cuda"))):
        assert H.rms_norm(a, b, 1e-6) is NotImplemented
        if b.dtype == a.dtype:
            assert torch.equal(LO.rms_norm(a, b, 1e-6), torch.nn.functional.rms_norm(a, (a.shape[-1],), b, 1e-6))
    leaf = x.clone().requires_grad_()
    LO.rms_norm(leaf, w, 1e-6).sum().backward()
    assert leaf.grad is not None
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert H.rms_norm(x, w, 1e-6) is NotImplemented


@pytest.mark.parametrize("W", [1024, 1032, 2048, 2056, 4096])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_a_row_stays_by_itself(W, dtype):
    """Rows of one wavefront and of four, of one unit a lane and of two: each what it is alone, beside rows that are zero and not numbers."""
    from jacobiforcing_amd import layer_ops as LO
    W = W if dtype == torch.bfloat16 else W // 2
    g = torch.Generator(device="cuda").manual_seed(W)
    x, w = torch.randn(9, W, generator=g, device="cuda").to(dtype), torch.randn(W, generator=g, device="cuda").to(dtype)
    x[2], x[5, W - 1], x[7, 0] = 0, float("nan"), float("inf")
    got = LO._host().rms_norm(x, w, 1e-6)
    assert got is not NotImplemented
    for r in range(9):
        assert torch.equal(got[r].nan_to_num(7.0), LO._host().rms_norm(x[r:r + 1], w, 1e-6)[0].nan_to_num(7.0)), r
        assert bool(got[r].isnan().all()) == (r == 5) and (r in (5, 7) or bool(got[r].isfinite().all())), r
