"""History tables that touch most of a row's vocabulary, on the sliced path:
a row's workspace holds the touched values of every kind of row up to the
point where they no longer fit, and beyond it the row is handed over
(sampling.py:48-106)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from deepseekrpc_amd import _native as N
from test_gpu_wide import PEN, rows_of, sample

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [16384, 20001, 33000])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("full", [False, True])
def test_tables_of_most_tokens(V, dtype, full):
    """The distinct tokens of a 16,384-token history, and nearly the whole vocabulary."""
    rng = np.random.default_rng(V)
    pols = [dict(p, **PEN) for p in (dict(top_k=50, top_p=0.9), dict(temperature=0.0), dict(top_p=0.9), dict(min_p=0.05), dict(),
                                     dict(top_k=1000, temperature=0.7), dict(temperature=0.0, top_k=4))]
    B = len(pols)
    x = rows_of(rng, B, V, "spiked", dtype)
    counts = np.zeros((B, V), np.int32)
    for r in range(B):
        at = rng.choice(V, int(0.97 * V) if full else int(V * -np.expm1(-16384 / V)), replace=False)
        counts[r, at] = rng.integers(1, 5, at.size)
    bias = [{5: 1.0, V - 1: -1.0}] * B  # keeps bf16 rows off the register kernel
    flags = sample(x, pols, rng.random(B), dtype, 1, counts, counts // 2, bias)
    assert full or (flags & N.FLAG_SPLIT).all(), [hex(int(f)) for f in flags]
