"""Top-k rows on the sliced path whose group prefixes cannot bound the
candidates: logits nearly equal or far from zero, ties at the k-th value, and
a top-k near the number of 16-token groups or of finite tokens
(sampling.py:86-106)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from deepseekrpc_amd import _native as N
from deepseekrpc_amd import workloads
from test_gpu_wide import PEN, histories, rows_of, sample

pytestmark = pytest.mark.gpu

POLICIES = [dict(top_k=20, temperature=5.0, top_p=0.95), dict(top_k=1024, top_p=0.99), dict(top_k=1), dict(top_k=1000, temperature=0.3),
            dict(top_k=500, min_p=0.5), dict(top_k=700, temperature=1.5, min_p=0.01, top_p=0.9)]


@pytest.mark.parametrize("V", [8192, 16399, 40000, 129280])
@pytest.mark.parametrize("kind,offset", [("flat", 20.0), ("flat", 80.0), ("normal", 150.0), ("spiked", -80.0), ("normal", 0.0)])
def test_close_rows_keep_the_path(V, kind, offset):
    rng = np.random.default_rng(V + int(offset))
    B = len(POLICIES)
    x = rows_of(rng, B, V, kind, torch.float32) + np.float32(offset)
    counts, gens = histories(rng, B, V, min(4000, V // 4))
    biases = [{int(t): float(rng.uniform(-1e-3, 1e-3)) for t in rng.choice(V, 30, replace=False)} for _ in range(B)]
    allowed = rng.random((B, V)) < 0.9
    pen = dict(repetition_penalty=1.0, presence_penalty=1e-4, frequency_penalty=1e-5) if kind == "flat" else PEN
    pols = [dict(p, **pen) for p in POLICIES]
    for al in (None, allowed):
        flags = sample(x, pols, rng.random(B), torch.float32, 1, counts, gens, biases, al)
        assert (flags & N.FLAG_SPLIT).all(), [hex(int(f)) for f in flags]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_few_finite_tokens(dtype):
    """Finite tokens in few groups or in as many as they are, more and fewer than k; tie groups at the k-th value."""
    rng = np.random.default_rng(7)
    V, B = 20000, 6
    x = rows_of(rng, B, V, "normal", dtype)
    allowed = np.zeros((B, V), bool)
    for r, n in enumerate((1, 3, 300, 900, 1500, 4000)):
        allowed[r, rng.choice(V, n, replace=False) if r % 2 else np.arange(V - n, V)] = True
    x[4] = workloads.bf16_round(np.round(x[4]).astype(np.float32))
    pols = [dict(top_k=k, **PEN) for k in (5, 1024, 1024, 1000, 700, 1024)]
    counts, gens = histories(rng, B, V, 3000)
    flags = sample(x, pols, rng.random(B), dtype, 1, counts, gens, None, allowed)
    on = [p["top_k"] <= n for p, n in zip(pols, (1, 3, 300, 900, 1500, 4000))]  # fewer than k: handed over
    assert ((flags & N.FLAG_SPLIT) != 0).tolist() == on, [hex(int(f)) for f in flags]
