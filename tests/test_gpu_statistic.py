"""The FP32 four-state branch statistic, pattern by pattern: with the weight on one pattern d logL/dP is
that pattern's alone, whichever lane, tile and wave of a workgroup holds it."""
import numpy as np
import pytest
import torch

from oracle import pruning as opruning
from test_walk4_program import _tree

pytestmark = pytest.mark.gpu
F64 = torch.float64


@pytest.mark.parametrize("dense", [False, True])
@pytest.mark.parametrize("C", [1, 2, 3, 4])
def test_each_pattern_counts_once(gpu, C, dense):
    """Tolerance: that of the other FP32 four-state gradients (1e-5 norm-wise)."""
    from torchtree_amd import likelihood as hl

    T, N = 7, 330  # two workgroups, the second with one whole and one ragged tile
    rng = np.random.default_rng(C)
    post = _tree("random", T)
    rows = np.vstack((np.eye(4), np.ones((1, 4))))[rng.integers(0, 5, (T, N))]
    if dense:
        rows = rows * rng.uniform(0.2, 1.0, rows.shape) + 0.01
    tips = [torch.tensor(r.T.copy()).float().double() for r in rows] + [None] * (T - 1)
    mats = rng.uniform(0.1, 1.0, (1, 2 * T - 2, C, 4, 4)) + 4 * np.eye(4)
    mats = torch.tensor(mats / mats.sum(-1, keepdims=True)).float().double()
    freqs, props = torch.full((1, 4), 0.25, dtype=F64), torch.full((C, 1, 1), 1.0 / C, dtype=F64)
    for n in (0, 3, 4, 15, 16, 31, 32, 61, 63, 64, 200, 255, 256, 319, 320, 329):
        print(f"case: statistic C={C} dense={dense} pattern {n}", flush=True)
        weights = torch.zeros(N, dtype=F64)
        weights[n] = 3.0
        m = mats.clone().requires_grad_(True)
        # (the oracle sees that pattern alone: it weighs log 0 of others by 0 as well)
        opruning.treelik_discrete_rescaled([t if t is None else t[:, n:n + 1] for t in tips],
                                           weights[n:n + 1], post, m, freqs, props).sum().backward()
        f32 = dict(device=gpu, dtype=torch.float32)
        g = mats.to(**f32).requires_grad_(True)
        hl.calculate_treelikelihood_discrete([t if t is None else t.to(gpu) for t in tips],
                                             weights.to(gpu), post, g, freqs.to(**f32),
                                             props.to(**f32)).sum().backward()
        assert float((g.grad.double().cpu() - m.grad).norm() / m.grad.norm()) < 1e-5, n
