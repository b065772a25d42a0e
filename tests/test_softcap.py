"""The logits' soft cap: in place on floats as before, and from bfloat16 in one pass, at lengths beside fours and workgroups and from borders beside them; the same bits as after a conversion."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 4, 1023, 1024, 1025, 70001])
@pytest.mark.parametrize("skip", [0, 1, 4])
def test_soft_cap(n, skip):
    from jacobiforcing_amd import layer_ops as LO
    g = torch.Generator(device="cuda").manual_seed(n)
    z = (torch.randn(n + skip, generator=g, device="cuda") * 40).bfloat16()[skip:]
    z[-1] = float("inf")
    f = torch.empty(n + skip, device="cuda")[skip:].copy_(z)
    got = LO.softcap_float(z, 30.0)
    assert LO.softcap(f, 30.0) is f and torch.equal(f, got) and got.dtype == torch.float32
    # a division, tanhf (2 units in the last place) and a product
    assert float((got.double() - 30.0 * torch.tanh(z.double() / 30.0)).abs().max()) <= 30.0 * 4 * 2.0 ** -24
