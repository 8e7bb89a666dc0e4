"""The verifier reads one allow mask per target row (dsr_verify_args_t); a
tensor of any other number of masks is refused before a launch, which would
read past its end."""
from __future__ import annotations

import pytest
import torch

from deepseekrpc_amd import batch

pytestmark = pytest.mark.gpu


def call(mask):
    R, K, V = 2, 3, 8192
    g = torch.Generator(device="cuda").manual_seed(1)
    t = torch.randn(R, K + 1, V, generator=g, device="cuda")
    d = t[:, :K].contiguous()
    return batch.verify_drafts(t, d, d.argmax(-1).to(torch.int32).contiguous(), batch.policy_tensor([dict(top_k=5)] * R, "cuda"),
                               torch.zeros(R, K, dtype=torch.float64, device="cuda"), torch.zeros(R, dtype=torch.float64, device="cuda"),
                               torch.full((R,), 10, dtype=torch.int32, device="cuda"), allow_bits=mask)


@pytest.mark.parametrize("shape,dtype", [((2, 256), torch.int32), ((2, 3, 256), torch.int32), ((2, 4, 256), torch.int16),
                                         ((2, 4, 256), torch.int64)])
def test_wrong_masks_are_refused(shape, dtype):
    with pytest.raises(ValueError, match="allow_bits"):
        call(torch.full(shape, -1, dtype=dtype, device="cuda"))


@pytest.mark.parametrize("shape", [(2, 4, 256), (8, 256), (2, 4, 300)])
def test_a_mask_per_target_row_is_taken(shape):
    res = call(torch.full(shape, -1, dtype=torch.int32, device="cuda"))
    assert res.status.tolist() == [0, 0] and res.accepted.tolist() == [3, 3]
