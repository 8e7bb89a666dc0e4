"""Kept bits of whole rows without a history or bias on the sliced path: every
finite allowed token's bit, whichever wave of a slice's workgroup wrote its
word first (sampling.py:79-106; the filters change probabilities, not the
top-k set)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from deepseekrpc_amd import _native as N
from deepseekrpc_amd import batch

pytestmark = pytest.mark.gpu


# The last word, vector and slice whole or cut short; enough workgroups that their waves start apart.
@pytest.mark.parametrize("V,rows", [(16384, 300), (16385, 200), (40007, 128), (129280, 64)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("mask", [False, True])
def test_every_finite_token_is_kept(V, rows, dtype, mask):
    g = torch.Generator(device="cuda").manual_seed(V)
    x = torch.zeros(rows, V + 1, device="cuda", dtype=dtype)[:, :V]  # odd stride: bf16 rows come here too
    x.copy_(torch.randn(rows, V, generator=g, device="cuda"))
    x[torch.rand(rows, V, generator=g, device="cuda") < 0.02] = -float("inf")
    finite = (x > -float("inf")).cpu().numpy()
    bits = None
    if mask:
        allowed = np.random.default_rng(V).random((rows, V)) < 0.7
        finite &= allowed
        bits = torch.from_numpy(batch.pack_allow(allowed).view(np.int32)).cuda()
    pols = batch.policy_tensor([dict(temperature=1.1, **(dict(), dict(top_p=0.3), dict(min_p=0.5))[r % 3]) for r in range(rows)], "cuda")
    call = batch.PreparedSample(x, pols, kept=True, allow_bits=bits)
    for _ in range(4):
        call.result.kept_bits.fill_(-1)
        res = call.launch()
        assert not (res.flags & N.FLAG_GENERAL).any() and (res.status == 0).all()
        kept = batch.unpack_bits(res.kept_bits.cpu().numpy().view(np.uint32), V)
        np.testing.assert_array_equal(kept, finite)
