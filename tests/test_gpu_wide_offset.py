"""Rows whose logits share an offset on the sliced path.  The law depends on
v - max alone (sampling.py:86-106), and so must the path a row takes; rows
whose logits nearly equal each other may be handed over, and are decided alike."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from deepseekrpc_amd import _native as N
from deepseekrpc_amd import workloads
from test_gpu_wide import PEN, histories, rows_of, sample

pytestmark = pytest.mark.gpu

POLICIES = [dict(top_p=0.9), dict(temperature=0.7, top_p=0.95), dict(min_p=0.05), dict(temperature=1.3, top_p=0.8, min_p=0.02),
            dict(top_p=0.0), dict(min_p=1.0), dict(temperature=2.5, top_p=0.6), dict(temperature=5.0, top_p=0.999), dict(min_p=0.5, top_p=0.5)]


@pytest.mark.parametrize("offset", [-150.0, -80.0, 20.0, 70.0])
@pytest.mark.parametrize("V", [16385, 40007, 129280])
def test_a_common_offset_keeps_the_path(V, offset):
    rng = np.random.default_rng(V + int(offset) + 1000)
    B = len(POLICIES)
    x = np.concatenate([rows_of(rng, 1, V, ("spiked", "normal")[r % 2], torch.float32) for r in range(B)]) + np.float32(offset)
    allowed = rng.random((B, V)) < 0.8
    u = rng.random(B)
    flags = sample(x, POLICIES, u, torch.float32, 1)
    assert (flags & N.FLAG_SPLIT).all(), [hex(int(f)) for f in flags]
    counts, gens = histories(rng, B, V, min(3000, V // 5))
    biases = [{int(t): float(rng.uniform(-3, 3)) for t in rng.choice(V, 20, replace=False)} for _ in range(B)]
    flags = sample(x, [dict(p, **PEN) for p in POLICIES], u, torch.float32, 3, counts, gens, biases, allowed)
    assert (flags & N.FLAG_SPLIT).all(), [hex(int(f)) for f in flags]


@pytest.mark.parametrize("V", [16384, 24575, 129280])
@pytest.mark.parametrize("width,offset", [(1e-3, 2e-3), (0.05, 8.0), (30.0, -500.0)])
def test_close_rows(V, width, offset):
    rng = np.random.default_rng(V + int(1000 * width))
    B = len(POLICIES)
    x = (rng.uniform(-width, width, (B, V)) + offset).astype(np.float32)
    flags = sample(x, POLICIES, rng.random(B), torch.float32, 1)
    if width > 1.0:
        assert (flags & N.FLAG_SPLIT).all(), [hex(int(f)) for f in flags]


@pytest.mark.parametrize("offset", [0.0, 12.0])
def test_bf16_rows(offset):
    """bf16 values tie by the hundred: rows are handed over where a tie group outgrows the list, and decided alike."""
    rng = np.random.default_rng(4)
    B, V = len(POLICIES), 30000
    x = rows_of(rng, B, V, "normal", torch.bfloat16)
    x = workloads.bf16_round((x + np.float32(offset)).astype(np.float32))
    counts, gens = histories(rng, B, V, 3000)
    sample(x, [dict(p, **PEN) for p in POLICIES], rng.random(B), torch.bfloat16, 1, counts, gens)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_unfiltered_rows_crowded_into_one_block(dtype):
    """No filter, penalised: the slices' sums decide the row however its tokens lie."""
    rng = np.random.default_rng(12)
    V = 20001
    x = np.concatenate([rows_of(rng, 1, V, "flat", torch.float32) + np.float32(0.003), rows_of(rng, 1, V, "normal", torch.float32),
                        rows_of(rng, 1, V, "normal", torch.float32) + np.float32(90.0)]).astype(np.float32)
    if dtype == torch.bfloat16:
        x = workloads.bf16_round(x)
    counts, gens = histories(rng, 3, V, 4000)
    bias = [{5: 0.5, V - 1: -1.0}] * 3  # keeps bf16 rows off the register kernel
    flags = sample(x, [dict(PEN), dict(PEN, temperature=0.6), dict(PEN)], rng.random(3), dtype, 1, counts, gens, bias)
    assert (flags & N.FLAG_SPLIT).all(), [hex(int(f)) for f in flags]
