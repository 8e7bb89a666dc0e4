"""Top-p cuts among tokens whose masses the sliced path's fixed-point sums
(steps of 2^-45) resolve to a few percent only: those sums may point a sub-bin
too low, and the float64 masses must not let that decide (sampling.py:97-102)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from test_gpu_wide import sample

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V,n", [(16384, 1800), (40000, 4000)])
def test_a_cut_among_tiny_masses(V, n):
    """One token of nearly all the mass and n of about 1e-12: the boundary lies among those."""
    rng = np.random.default_rng(V)
    B = 32
    x = np.full((B, V), -60.0, np.float32)
    pols = []
    for r in range(B):
        at = rng.choice(V, n + 1, replace=False)
        x[r, at[0]] = 0.0
        x[r, at[1:]] = rng.normal(-27.6, 0.3, n)
        e = np.exp(np.sort(x[r].astype(np.longdouble))[::-1])
        cum = np.cumsum(e)
        m = int(rng.integers(n // 4, n))
        pols.append(dict(top_p=float((cum[m - 1] - e[m - 1] / 2) / cum[-1])))  # the middle of the m-th token's mass
    sample(x, pols, rng.random(B), torch.float32, 1)
