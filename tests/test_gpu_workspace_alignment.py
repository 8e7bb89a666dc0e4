"""A workspace that is only 8-byte aligned, which dsr_sample_rows accepts,
gives the results of an aligned one; the sliced path, which reads its
workspace 16 bytes at a time, leaves such calls to the other paths."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from deepseekrpc_amd import _native as N
from deepseekrpc_amd import batch
from test_gpu_wide import device_logits, rows_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,V,pol", [(torch.float32, 20000, dict(top_p=0.9)), (torch.float32, 40000, dict(top_k=40)),
                                         (torch.bfloat16, 9000, dict(top_k=40, top_p=0.9)), (torch.bfloat16, 16391, dict())])
def test_eight_byte_aligned_workspace(dtype, V, pol):
    rng = np.random.default_rng(V)
    B = 5
    x = device_logits(rows_of(rng, B, V, "normal", dtype), dtype, 1)
    call = batch.PreparedSample(x, batch.policy_tensor([pol] * B, "cuda"), uniforms=torch.from_numpy(rng.random(B)).cuda(), probs="f64")
    torch.cuda.synchronize()
    want = [getattr(call.result, f).clone() for f in ("tokens", "consumed", "status", "probs")]
    assert not (call.result.flags & N.FLAG_GENERAL).any()
    need = N.load().dsr_sample_workspace_bytes(B, V)
    buf = torch.empty(need + 16, dtype=torch.uint8, device="cuda")
    call.args.workspace, call.args.workspace_bytes = buf.data_ptr() + 8, need
    assert call.args.workspace % 16 == 8
    res = call.launch()
    torch.cuda.synchronize()
    for w, f in zip(want[:3], ("tokens", "consumed", "status")):
        assert torch.equal(w, getattr(res, f)), f
    torch.testing.assert_close(res.probs, want[3], rtol=1e-12, atol=0.0)
    if V < 16384 and dtype == torch.bfloat16:  # no other path than the general one takes these rows
        assert (res.flags & N.FLAG_GENERAL).all()
