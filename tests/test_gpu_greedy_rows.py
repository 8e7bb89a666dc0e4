"""Greedy rows with a history in a large bf16 batch: decided in a launch of
their own (or left by it to the full-vocabulary kernel), whatever their order
among the sampled rows, as in a batch small enough for one launch
(sampling.py:48-90)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from deepseekrpc_amd import batch
from oracle import sampling_oracle as O

pytestmark = pytest.mark.gpu

PEN = dict(repetition_penalty=1.2, presence_penalty=0.5, frequency_penalty=0.25)


@pytest.mark.parametrize("V,rows", [(8, 257), (520, 300), (8200, 288), (129280, 261)])
@pytest.mark.parametrize("mask", [False, True])
def test_large_batches_decide_as_small_ones(V, rows, mask):
    rng = np.random.default_rng(V + rows + mask)
    x = rng.normal(0, 2, (rows, V)).astype(np.float32)
    x[3::7] = np.round(x[3::7])                               # ties, some of them at the maximum
    x[5::31] = -np.abs(x[5::31])
    x[5::31, V // 2] = 0.0                                    # a maximum of zero: handed over
    x[11, V - 1] = np.nan
    x[12, 0] = np.inf
    x[13] = -np.inf
    logits = torch.from_numpy(x).to(torch.bfloat16)
    pols = [dict(PEN, **(dict(temperature=0.0) if r % 3 != 1 else dict(top_p=0.9))) for r in range(rows)]
    pols[17] = dict(temperature=0.0, top_k=3)                 # a greedy row with a top-k
    hist = [rng.integers(0, V, int(rng.integers(0, min(V // 2, 600)))) for _ in range(rows)]
    hist[20] = np.argsort(-x[20])[: V // 4]                   # the likeliest tokens
    hist[21] = np.arange(V - V // 4)                          # more than the workspace row holds
    table = batch.HistoryTable.from_token_lists([h.tolist() for h in hist], device="cuda")
    allowed = rng.random((rows, V)) < 0.8 if mask else None
    bits = torch.from_numpy(batch.pack_allow(allowed).view(np.int32)).cuda() if mask else None
    u = torch.from_numpy(rng.random(rows)).cuda()
    d = logits.cuda()
    got = batch.sample_rows(d, batch.policy_tensor(pols, "cuda"), uniforms=u, history=table, allow_bits=bits)
    seen = logits.float().numpy()
    for lo in range(0, rows, 128):                            # the same rows, few enough for the one launch
        hi = min(lo + 128, rows)
        part = batch.HistoryTable.from_token_lists([h.tolist() for h in hist[lo:hi]], device="cuda")
        want = batch.sample_rows(d[lo:hi].contiguous(), batch.policy_tensor(pols[lo:hi], "cuda"), uniforms=u[lo:hi].contiguous(),
                                 history=part, allow_bits=bits[lo:hi].contiguous() if mask else None)
        for f in ("tokens", "consumed", "status", "flags"):
            a, b = getattr(got, f)[lo:hi], getattr(want, f)
            assert torch.equal(a, b), (f, lo, torch.nonzero(a != b).flatten().tolist())
    for r in [0, 2, 3, 5, 11, 13, 17, 20, 21, rows - 1]:      # and the oracle's
        if pols[r]["temperature"] if "temperature" in pols[r] else 1.0:
            continue
        counts = np.bincount(hist[r], minlength=V).astype(np.int32)
        try:
            p = O.probabilities(seen[r], O.Policy(**pols[r]), counts, counts, {}, allowed[r] if mask else None)
            assert int(got.status[r]) == 0 and int(got.tokens[r]) == int(np.argmax(p)), r
        except O.OracleError as e:
            assert int(got.status[r]) != 0, (r, e)
