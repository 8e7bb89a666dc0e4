"""Large batches of the full-vocabulary kernel, whose sampled rows start before
its greedy ones and whose greedy rows may be decided in a launch of their own:
every row as in a batch of its own kind small enough for one round
(sampling.py:48-128)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from deepseekrpc_amd import batch

pytestmark = pytest.mark.gpu

PEN = dict(repetition_penalty=1.2, presence_penalty=0.5, frequency_penalty=0.25)
FIELDS = ("tokens", "consumed", "status", "flags")


def compare(got, part, rows):
    for lo in range(0, rows, 200):
        hi = min(lo + 200, rows)
        want = part(lo, hi)
        for f in FIELDS:
            a, b = getattr(got, f)[lo:hi], getattr(want, f)
            assert torch.equal(a, b), (f, lo, torch.nonzero(a != b).flatten().tolist())


# Around the sizes where the order, the greedy launch and the order's limit begin; shares of greedy rows on
# both sides of that launch's rule.
@pytest.mark.parametrize("rows,share", [(257, 0.5), (767, 0.9), (768, 0.9), (768, 0.01), (1024, 0.5), (1500, 0.97), (4096, 0.6), (4097, 0.5)])
def test_penalised_rows(rows, share):
    rng = np.random.default_rng(rows)
    V = 520
    x = rng.normal(0, 2, (rows, V)).astype(np.float32)
    x[3::7] = np.round(x[3::7])                              # ties at the maximum
    x[5::31] = -np.abs(x[5::31])
    x[5::31, V // 2] = 0.0                                   # a maximum of zero: left to the full-vocabulary kernel
    x[11, V - 1], x[12, 0], x[13] = np.nan, np.inf, -np.inf
    d = torch.from_numpy(x).to(torch.bfloat16).cuda()
    pols = [dict(PEN, **(dict(temperature=0.0) if g else dict(top_p=0.9))) for g in rng.random(rows) < share]
    hist = [rng.integers(0, V, int(rng.integers(0, 200))).tolist() for _ in range(rows)]
    u = torch.from_numpy(rng.random(rows)).cuda()
    run = lambda lo, hi: batch.sample_rows(d[lo:hi].contiguous(), batch.policy_tensor(pols[lo:hi], "cuda"), uniforms=u[lo:hi].contiguous(),
                                           history=batch.HistoryTable.from_token_lists(hist[lo:hi], device="cuda"))
    compare(run(0, rows), run, rows)


@pytest.mark.parametrize("rows", [300, 1100])
def test_whole_rows_among_top_k_rows(rows):
    rng = np.random.default_rng(rows)
    V = 4096
    d = torch.from_numpy(rng.normal(0, 2, (rows, V)).astype(np.float32)).to(torch.bfloat16).cuda()
    kinds = [dict(top_p=0.9), dict(top_k=20, top_p=0.9), dict(temperature=0.0), dict(), dict(top_k=3)]
    pols = [kinds[int(k)] for k in rng.integers(0, 5, rows)]
    u = torch.from_numpy(rng.random(rows)).cuda()
    run = lambda lo, hi: batch.sample_rows(d[lo:hi].contiguous(), batch.policy_tensor(pols[lo:hi], "cuda"), uniforms=u[lo:hi].contiguous())
    compare(run(0, rows), run, rows)
