"""Filtered and conditioned speculative requests on the sliced path against
the NumPy oracle, at the slice edges of its vocabulary range, for every
request kind it decides and the ones it hands to the general path
(sampling.py:255-319)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from deepseekrpc_amd import _native as N
from deepseekrpc_amd import batch
from oracle import sampling_oracle as O
from test_gpu_rng import verify_device_vs_host
from test_gpu_verify_general import STOP, _run

pytestmark = pytest.mark.gpu

TOPK = [dict(top_k=50, top_p=0.9, temperature=0.8), dict(top_k=1, temperature=0.6), dict(top_k=1000, min_p=0.01),
        dict(top_k=70, temperature=1.3), dict(top_k=8, top_p=0.5), dict(top_k=20, temperature=0.0)]
WHOLE = [dict(top_p=0.9, temperature=0.7), dict(top_p=0.4), dict(min_p=0.05), dict(top_p=0.8, min_p=0.02, temperature=1.2),
         dict(top_p=1e-9), dict(top_p=0.999, temperature=0.5)]
MIXED = TOPK[:3] + WHOLE[:3] + [dict(), dict(top_k=2000), dict(temperature=0.0), dict(top_p=0.0, top_k=0)]


def _plain(V, policies, K, dtype, seed, spoil=(), hints=None):
    rng = np.random.default_rng(seed)
    dev, R = "cuda", 2 * len(policies)
    pols = [dict(policies[r % len(policies)]) for r in range(R)]
    tgt = rng.normal(0, 2, (R, K + 1, V)).astype(np.float32)
    drf = (tgt[:, :K] + rng.normal(0, 0.4, (R, K, V))).astype(np.float32)
    drf[1] = tgt[1, :K]                                       # equal rows: every weight of a correction is 0
    tgt, drf = torch.from_numpy(tgt).to(dtype), torch.from_numpy(drf).to(dtype)
    for r, j in spoil:
        tgt[r, j, V - 1] = float("nan")
    st, sd = tgt.float().numpy(), drf.float().numpy()
    ids = np.zeros((R, K), np.int32)
    for r in range(R):
        pol = O.Policy(**pols[r])
        for j in range(K):
            row = st[r, j] if pol.temperature == 0 else sd[r, j]
            if pol.temperature == 0:
                drf[r, j] = tgt[r, j]
                sd[r, j] = st[r, j]
            try:
                ids[r, j] = O.categorical(O.probabilities(row, pol), float(rng.random()))[0]
            except O.OracleError:
                ids[r, j] = int(rng.integers(0, V))
    if K:
        ids[2 % R, 0] = int(np.argmin(sd[2 % R, 0]))           # outside a cut: no proposal mass
    lim = np.asarray([(10, 1, 2, 3)[r % 4] if r % 3 == 0 else 10 for r in range(R)], np.int32)
    ua, ut = rng.random((R, K)), rng.random(R)
    uad, utd = torch.from_numpy(ua).to(dev), torch.from_numpy(ut).to(dev)
    res = batch.verify_drafts(tgt.to(dev), drf.to(dev), torch.from_numpy(ids).to(dev), batch.policy_tensor(pols, dev), uad, utd,
                              torch.from_numpy(lim).to(dev), hints=hints)
    torch.cuda.synchronize()
    for r in range(R):
        ref = O.verify(st[r], sd[r], list(ids[r]), O.Policy(**pols[r]), ua[r], float(ut[r]), output_limit=int(lim[r]))
        n = int(res.count[r])
        got = (int(res.status[r]), int(res.accepted[r]), tuple(res.ids[r, :n].tolist()),
               None if int(res.pending[r]) < 0 else int(res.pending[r]), STOP[int(res.stop[r])],
               int(res.used_accept[r]), int(res.used_target[r]))
        if ref.status:
            want = (ref.status, 0, (), None, None, 0, 0)
        else:
            want = (0, ref.accepted, ref.output_ids, ref.pending, ref.stop, ref.used_accept, ref.used_target)
        assert got == want, (r, pols[r], got, want, ref.margin)
    return res


@pytest.mark.parametrize("V,dtype", [(8192, torch.float32), (8193, torch.bfloat16), (16391, torch.float32),
                                     (24576, torch.bfloat16)])
@pytest.mark.parametrize("kind", ["topk", "whole", "mixed"])
def test_filtered_requests(V, dtype, kind):
    res = _plain(V, dict(topk=TOPK, whole=WHOLE, mixed=MIXED)[kind], 3, dtype, seed=V)
    assert res.args.hints == dict(topk=N.HINT_TOPK_ALL, whole=N.HINT_WHOLE_SOME, mixed=0)[kind]
    if kind == "mixed":
        _plain(V, MIXED, 3, dtype, seed=V, hints=N.HINT_WHOLE_SOME)
        _plain(V, MIXED, 3, dtype, seed=V, hints=N.HINT_TOPK_ALL)
    assert (res.status == 0).sum() >= 8


@pytest.mark.parametrize("kind", ["topk", "mixed"])
def test_filtered_requests_full_vocab(kind):
    _plain(129280, dict(topk=TOPK, mixed=MIXED)[kind], 2, torch.float32, seed=5, hints=N.HINT_WHOLE_SOME)


@pytest.mark.parametrize("K", [0, 1, 5])
def test_draft_counts(K):
    _plain(8200, MIXED, K, torch.float32, seed=40 + K, hints=N.HINT_WHOLE_SOME)


def test_invalid_rows_are_reported_as_they_are_reached():
    """A NaN in the first, a middle and the bonus target row: the request is
    built in full, and fails only where the chain reaches the row."""
    res = _plain(8192, TOPK[:5] + WHOLE[:5], 3, torch.float32, seed=77,
                 hints=N.HINT_WHOLE_SOME, spoil=[(0, 0), (3, 1), (4, 3), (5, 0), (7, 1), (8, 3)])
    assert int(res.status[0]) == N.E_LOGITS and int(res.status[5]) == N.E_LOGITS


def test_hints_of_known_policies():
    hints = lambda p, plain=True: batch._verify_call_hints(batch.policy_array(p), 129280, plain)
    assert hints(TOPK) == N.HINT_TOPK_ALL and hints(WHOLE) == hints(TOPK + WHOLE) == N.HINT_WHOLE_SOME
    assert hints([dict(temperature=0.0), dict(top_k=9)]) == 0                        # the greedy one is fast
    assert hints([dict(temperature=0.0), dict(top_k=9)], False) == N.HINT_TOPK_ALL
    assert hints(WHOLE, False) == hints([dict(top_k=2000)]) == hints(WHOLE + [dict()]) == 0


@pytest.mark.parametrize("V,dtype", [(8192, torch.float32), (8199, torch.bfloat16), (24575, torch.float32)])
def test_conditioned_requests(V, dtype):
    outcome = _run(V, 18, 4, dtype, seed=311)
    assert sum(o[0] == 0 for o in outcome.values()) >= 10


def test_device_draws():
    R, K, V = 12, 3, 16400
    g = torch.Generator(device="cuda").manual_seed(3)
    tgt = 2 * torch.randn(R, K + 1, V, generator=g, device="cuda")
    drf = (tgt[:, :K] + 0.5 * torch.randn(R, K, V, generator=g, device="cuda")).contiguous()
    pols = (TOPK[:1] + WHOLE[:1] + TOPK[3:4] + WHOLE[3:4]) * 3
    ids = batch.sample_rows(drf.reshape(R * K, V), [p for p in pols for _ in range(K)],
                            uniforms=torch.rand(R * K, generator=g, device="cuda", dtype=torch.float64)).tokens
    limit = torch.full((R,), 10, dtype=torch.int32, device="cuda")
    got = verify_device_vs_host(tgt, drf, ids.reshape(R, K).contiguous(), pols, limit, 910)
    assert int(got.used_accept.sum()) > R and int(got.used_target.sum()) > 0
