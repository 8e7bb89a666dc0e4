"""Rows whose mask or logits leave whole 8,192-token slices without a finite
token, in a workspace full of NaN patterns: what those slices leave unwritten
must not reach the row's decision or send it to the general path
(sampling.py:75-106)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from deepseekrpc_amd import _native as N
from deepseekrpc_amd import batch
from oracle import sampling_oracle as O
from test_gpu_wide import device_logits, rows_of

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("V", [16385, 24577, 129280])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_slices_without_a_finite_token(V, dtype):
    rng = np.random.default_rng(V)
    pols = [dict(top_p=0.9), dict(top_p=0.8, min_p=0.02, temperature=1.3), dict(min_p=0.05), dict(), dict(top_k=20), dict(temperature=0.0)]
    B = len(pols)
    x = rows_of(rng, B, V, "spiked", dtype)
    allowed = np.ones((B, V), bool)
    allowed[:, 8192:] = False          # the first slice is left
    allowed[3:, 16384:16390] = True    # and a few tokens of a later one
    x[1, 8192:] = -np.inf              # nothing finite under the mask either
    u = rng.random(B)
    need = batch.N.load().dsr_sample_workspace_bytes(B, V)
    ws = batch.Workspace()
    call = batch.PreparedSample(device_logits(x, dtype, 1), batch.policy_tensor(pols, DEV), probs="f64", workspace=ws,
                                uniforms=torch.from_numpy(u).to(DEV),
                                allow_bits=torch.from_numpy(batch.pack_allow(allowed).view(np.int32)).to(DEV))
    buf = call.result.keep[7]
    assert buf.numel() * buf.element_size() >= need
    buf.view(torch.uint8).fill_(255)
    res = call.launch()
    torch.cuda.synchronize()
    for r in range(B):
        ref = O.sample_row(x[r], O.Policy(**pols[r]), float(u[r]), None, None, None, allowed[r])
        assert (int(res.status[r]), int(res.tokens[r])) == (0, ref.token), r
        np.testing.assert_allclose(res.probs[r].cpu().numpy(), ref.probs, rtol=1e-12, atol=1e-300)
    assert not (res.flags & N.FLAG_GENERAL).any(), res.flags.tolist()
