"""The bonus token of a filtered row whose 16 draws all collide with its proposal: the segments' masses lead to it (rs_masked_argmax_full), against the row-by-row restatement."""
import numpy as np
import pytest
import torch

from jacobiforcing_amd import _native as N
from jacobiforcing_amd import ops
from tests.backends import device_for, use_backend
from tests.test_kernels import _assert_rs_equal

pytestmark = pytest.mark.gpu


# kept ids over all segments, over a few, one beside the proposal, none but the proposal; equal values in several segments; one segment, beside a whole tile
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("coarse", [False, True], ids=["distinct", "tied"])
@pytest.mark.parametrize("V,top_k,top_p", [(152064, 50, 0.0), (152064, 50, 0.985), (152064, 2, 0.0), (152064, 0, 0.9), (152064, 400, 0.999), (32000, 7, 0.0), (2047, 50, 0.99), (50, 20, 0.0)])
def test_masked_argmax_of_filtered_rows(dtype, coarse, V, top_k, top_p):
    B, L = 6, 4
    g = torch.Generator().manual_seed(V + top_k)
    draft = torch.randint(0, V, (B, L), generator=g)
    draft[0, 1:], draft[1, 1:] = V - 1, 0                                # the proposal in the last segment, in the first
    logits = torch.randn(B, L - 1, V, generator=g) * 2
    if coarse:
        logits = torch.round(logits)
    # the proposal holds 0.97 of what the filters keep
    kept = logits.topk(min(top_k or V, V), -1).values
    logits.scatter_(2, draft[:, 1:].unsqueeze(-1), (torch.logsumexp(kept, -1) + float(np.log(0.97 / 0.03))).unsqueeze(-1))
    n = 4 * B * L * 16
    unis, bonus = torch.full((n,), 0.9995), torch.randint(0, 1 << 24, (n,), generator=g).float() / float(1 << 24)
    pads = torch.randint(0, V, (n,), generator=g)
    out = {}
    for backend in ("hip", "hostsim"):
        with use_backend(backend):
            dev = device_for(backend)
            st = ops.RsStepper(B, L, dev, pads, unis, bonus)
            rows, toks, nd = st.step(draft.to(dev), logits.to(dtype).to(dev), 1.0, None, [L] * B, [1, 2, 3], top_k, top_p)
            out[backend] = (rows.copy(), toks.copy(), nd.cpu().numpy().copy(), st.cursors.cpu().tolist())
    _assert_rs_equal(out["hip"], out["hostsim"], B)
    draws = out["hostsim"][0][:, N.RS_FIELDS.index("n_bonus_draws")]
    assert top_p == 0.9 or (draws == 16).sum() >= 1                      # (there the proposal alone is kept, and accepted)
