"""Hints choose launches only: on batches the sliced path takes, every row is
decided, and alike, under each combination of DSR_HINT_WHOLE_SOME,
DSR_HINT_WHOLE_ALL and DSR_HINT_TOPK_ALL, whatever the rows are."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from deepseekrpc_amd import _native as N
from deepseekrpc_amd import batch
from oracle import sampling_oracle as O
from test_gpu_wide import device_logits, histories, rows_of

pytestmark = pytest.mark.gpu
DEV = "cuda"

POLICIES = [dict(temperature=0.7, top_k=50, top_p=0.9), dict(top_p=0.9), dict(temperature=0.0), dict(top_k=2000),
            dict(), dict(top_k=8, min_p=0.02), dict(min_p=0.05), dict(top_k=1024)]
COMBINATIONS = [0, N.HINT_WHOLE_SOME, N.HINT_WHOLE_ALL, N.HINT_WHOLE_SOME | N.HINT_WHOLE_ALL, N.HINT_TOPK_ALL,
                N.HINT_TOPK_ALL | N.HINT_WHOLE_SOME, N.HINT_TOPK_ALL | N.HINT_WHOLE_ALL,
                N.HINT_TOPK_ALL | N.HINT_WHOLE_SOME | N.HINT_WHOLE_ALL]


@pytest.mark.parametrize("dtype,V,pad,tables", [(torch.float32, 20000, 0, False), (torch.float32, 33000, 0, False),
                                                (torch.float32, 20000, 1, True), (torch.bfloat16, 16384, 0, True),
                                                (torch.bfloat16, 16384, 3, False)])
def test_every_combination_decides_every_row(dtype, V, pad, tables):
    rng = np.random.default_rng(V + pad)
    B = len(POLICIES)
    x = rows_of(rng, B, V, "spiked", dtype)
    u = rng.random(B)
    counts = histories(rng, B, V, 2000)[0] if tables else None
    biases = [{int(t): 1.5 for t in rng.choice(V, 9, replace=False)} for _ in range(B)] if tables else None
    pols = [dict(p, **(dict(repetition_penalty=1.2) if tables else {})) for p in POLICIES]
    logits, policies = device_logits(x, dtype, pad), batch.policy_tensor(pols, DEV)
    kw = {}
    if tables:
        kw = dict(history=batch.HistoryTable.from_dense(counts, counts, device=DEV),
                  bias=batch.BiasTable.from_dicts(biases, device=DEV))
    refs = [O.sample_row(x[r], O.Policy(**pols[r]), float(u[r]), counts[r] if tables else None,
                         counts[r] if tables else None, biases[r] if tables else None, None) for r in range(B)]
    for hints in COMBINATIONS:
        out = dict(tokens=torch.full((B,), -77, dtype=torch.int32, device=DEV),
                   consumed=torch.full((B,), 77, dtype=torch.uint8, device=DEV),
                   status=torch.full((B,), 77, dtype=torch.int32, device=DEV),
                   flags=torch.full((B,), 255, dtype=torch.uint8, device=DEV),
                   probs=torch.full((B, V), 7.0, dtype=torch.float64, device=DEV))
        res = batch.sample_rows(logits, policies, uniforms=torch.from_numpy(u).to(DEV), probs="f64", kept=True,
                                hints=hints, out=out, **kw)
        torch.cuda.synchronize()
        kept = batch.unpack_bits(res.kept_bits.cpu().numpy().view(np.uint32), V)
        for r, ref in enumerate(refs):
            got = (int(res.status[r]), int(res.tokens[r]), bool(res.consumed[r]))
            assert got == (0, ref.token, ref.consumed), (hints, r, got, ref.token)
            np.testing.assert_allclose(res.probs[r].cpu().numpy(), ref.probs, rtol=1e-12, atol=1e-300, err_msg=f"{hints} {r}")
            np.testing.assert_array_equal(kept[r], ref.topk_kept, err_msg=f"{hints} {r}")


def test_policies_rewritten_under_a_prepared_call():
    """A kept call's hints are those of its first policies; the tensor may be rewritten in place."""
    rng = np.random.default_rng(3)
    V, B = 20000, 6
    x = rows_of(rng, B, V, "spiked", torch.float32)
    u = rng.random(B)
    for first, then in (([dict(top_p=0.9)] * B, [dict(top_k=40)] * B), ([dict(top_k=40)] * B, [dict(top_p=0.9)] * B)):
        policies = batch.policy_tensor(first, DEV)
        call = batch.PreparedSample(device_logits(x, torch.float32, 1), policies, uniforms=torch.from_numpy(u).to(DEV))
        policies.copy_(batch.policy_tensor(then, DEV))
        call.result.tokens.fill_(-77)
        res = call.launch()
        torch.cuda.synchronize()
        want = [O.sample_row(x[r], O.Policy(**then[r]), float(u[r]), None, None, None, None).token for r in range(B)]
        assert res.tokens.tolist() == want and (res.status == 0).all()
