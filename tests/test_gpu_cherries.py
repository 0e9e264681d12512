"""The four-state FP32 gradient where both children of a node are cherries of small partials."""
import numpy as np
import pytest
import torch

from oracle import pruning as opruning

pytestmark = pytest.mark.gpu
F64 = torch.float64


@pytest.mark.parametrize("C", [1, 2, 3, 4])
@pytest.mark.parametrize("T", [4, 12])
def test_two_cherries_of_small_partials(gpu, T, C):
    """Tips of a cherry that differ across branches of 1e-25: its partial is 1e-25, and the product of
    two such is below what FP32 holds. Tolerance: that of the other FP32 gradients (1e-5 norm-wise)."""
    from torchtree_amd import likelihood as hl

    # quartets ((0,1),(2,3)) joined as a caterpillar
    post, nxt, prev = [], T, None
    for q in range(0, T, 4):
        post += [(nxt, q, q + 1), (nxt + 1, q + 2, q + 3), (nxt + 2, nxt, nxt + 1)]
        nxt += 3
        if prev is not None:
            post.append((nxt, prev, nxt - 1))
            nxt += 1
        prev = nxt - 1
    rng = np.random.default_rng(T + C)
    N, B = 67, 2 * T - 2
    codes = rng.integers(0, 4, (T, N))
    codes[1::2] = (codes[0::2] + rng.integers(1, 4, codes[0::2].shape)) % 4
    small = np.zeros(B, bool)
    small[:T] = True
    off = np.where(small, 1e-25, 0.05)[:, None, None, None] * rng.uniform(0.5, 1.0, (B, C, 4, 4))
    mats = torch.tensor(np.where(np.eye(4, dtype=bool), 1.0, off)[None]).float()
    tips = [torch.eye(4, dtype=F64)[torch.tensor(codes[t])].T.contiguous() for t in range(T)]
    weights = torch.ones(N, dtype=F64)
    freqs, props = torch.full((1, 4), 0.25), torch.full((C, 1, 1), 1.0 / C)
    ref_m = mats.double().requires_grad_(True)
    ref = opruning.treelik_discrete_rescaled(tips + [None] * (T - 1), weights, post, ref_m,
                                             freqs.double(), props.double())
    ref.sum().backward()
    m = mats.to(gpu).requires_grad_(True)
    got = hl.calculate_treelikelihood_discrete([t.to(gpu) for t in tips] + [None] * (T - 1),
                                               weights.to(gpu), post, m, freqs.to(gpu), props.to(gpu))
    got.sum().backward()
    assert float((got.detach().double().cpu() - ref.detach()).norm() / ref.detach().norm()) < 1e-6
    for part in (slice(0, T), slice(T, B)):  # (the gradients of the short branches are 1e24)
        a, b = m.grad[:, part].double().cpu(), ref_m.grad[:, part]
        assert float((a - b).norm() / b.norm()) < 1e-5
