"""What ``MultiblockBatch.results`` brings to the host: as many columns as the longest result, the same values as the whole list."""
import numpy as np
import pytest
import torch

from oracle import jacobi_oracle as O
from oracle.scripted_model import ScriptedModel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,n,lengths", [(1, 4, (60,)), (3, 16, (70, 200, 9)), (5, 8, (40, 41, 42, 43, 44))])
def test_results_are_the_whole_list(P, n, lengths):
    from jacobiforcing_amd import _native as N
    from jacobiforcing_amd import ops
    V, dev = 300, "cuda:0"
    models = [ScriptedModel(V, 11 + p, 70, lengths[p], eos_id=V - 1, eos_pos=None, reserved=(V - 2,)) for p in range(P)]
    batch = ops.MultiblockBatch(P, ops.MultiblockParams(n=n, K=2, r=0.5, n_gram_pool_size=4, eos_token_id=V - 1, pad_token_id=V - 2), dev)
    kvs = [m.prompt() for m in models]
    fwd = [(lambda m: (lambda kv, rows: [m.greedy_rows(kv[b], [rows[b]])[0] for b in range(len(rows))]))(m) for m in models]
    first = [O.mb_prefill(fwd[p], kvs[p], kvs[p][:1] * n)[0] for p in range(P)]
    d, cur, seen = batch.begin(torch.tensor(first), torch.tensor([len(k) for k in kvs], dtype=torch.int32)), [list(k) for k in kvs], set()

    def check(d):
        got, lens = batch.results(d), batch.desc_field(d, "ret_len").copy()
        whole = torch.zeros((P, batch.ret_cap), dtype=torch.int64, device=dev)
        N.check(N.lib().jf_mb_read_ret(batch.states.data_ptr(), batch.state_ints, P, whole.data_ptr(), batch.ret_cap, ops._stream(whole.device)))
        for p, row in enumerate(whole.cpu().tolist()):
            assert got[p]["ret"] == row[:lens[p]] and all(x == -1 for x in row[lens[p]:])
            assert (got[p]["kv_len"], got[p]["iters"], got[p]["next_token"]) == tuple(int(batch.desc_field(d, k)[p]) for k in ("kv_len", "iters", "next_token"))
        seen.add(int(lens.max()))

    check(d)
    while (pk := batch.pack(d)) is not None:
        ids, B, T = pk[0].cpu().numpy(), batch.desc_field(d, "B").copy(), batch.desc_field(d, "T").copy()
        logits, r0, rows_of = np.zeros((ids.shape[0], ids.shape[1], V), dtype=np.float32), 0, []
        for p in range(P):
            rows_of.append([ids[r0 + b, :T[p]].tolist() for b in range(B[p])])
            if B[p]:
                logits[r0:r0 + B[p], :T[p]] = models[p].logits_rows(cur[p], rows_of[p])
            r0 += B[p]
        d = batch.verify(torch.from_numpy(logits).to(dev))
        for p in range(P):
            if B[p]:
                src = int(batch.desc_field(d, "kv_src_row")[p]) if batch.desc_field(d, "kv_copy_len")[p] > 0 else 0
                cur[p] = cur[p] + rows_of[p][src][:int(batch.desc_field(d, "kv_len")[p]) - len(cur[p])]
        check(d)
        if batch.desc_field(d, "done").all():
            break
    assert max(seen) > 0
