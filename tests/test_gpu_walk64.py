"""The four-state FP64 post-order walk where it can go wrong: a tile's quarters and their edges, trees
that spill and trees that hold, every category count, coded and dense tips, one wave and four waves
per tile, with and without a gradient."""
import numpy as np
import pytest
import torch

from oracle import models as omodels
from oracle import pruning as opruning
from test_walk4_program import _tree

pytestmark = pytest.mark.gpu
F64 = torch.float64


@pytest.fixture(scope="module")
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch.device("cuda", 0)


CASES = [("random", 2, 1, 1, False, 1), ("random", 3, 16, 4, False, 2), ("caterpillar", 9, 17, 3, False, 1),
         ("balanced", 64, 63, 4, False, 1), ("balanced", 16, 65, 2, True, 3), ("random", 33, 130, 1, True, 1),
         ("random", 150, 100, 4, False, 1),
         # at least 768 tiles of all samples: one wave per tile
         ("balanced", 8, 49180, 1, False, 1), ("random", 9, 16400, 3, True, 3), ("random", 12, 24600, 2, False, 2),
         ("balanced", 8, 12301, 4, False, 4)]


@pytest.mark.parametrize("shape,T,N,C,dense,K", CASES)
def test_walk64(gpu, shape, T, N, C, dense, K):
    """Tolerances: those of the other FP64 tests (logL 1e-12, gradients 1e-10 norm-wise)."""
    print(f"case: FP64 walk {shape} T={T} N={N} C={C} dense={dense} K={K}", flush=True)
    from torchtree_amd import likelihood as hl

    rng = np.random.default_rng(T * N)
    post, B = _tree(shape, T), 2 * T - 2
    codes = (rng.integers(0, 4, size=(1, N)) + (rng.random((T, N)) < 0.3) * rng.integers(0, 4, (T, N))) % 4
    codes = np.where(rng.random((T, N)) < 0.05, 4, codes)
    table = np.vstack((np.eye(4), np.ones((1, 4))))
    tips = [torch.tensor(table[codes[t]].T.copy()) for t in range(T)]
    if dense:
        tips = [t * torch.tensor(rng.uniform(0.2, 1.0, t.shape)) + 0.01 for t in tips]
    weights = torch.tensor(rng.integers(1, 5, N).astype(float))
    freqs = torch.tensor(rng.dirichlet(np.full(4, 10.0)))
    q = omodels.gtr_q(torch.tensor(rng.gamma(2.0, 2.0, 6)), freqs)
    rates = torch.linspace(0.3, 2.0, C, dtype=F64) if C > 1 else torch.ones(1, dtype=F64)
    props = torch.full((C,), 1.0 / C, dtype=F64)
    bls = torch.tensor(rng.exponential(0.1, (K, B)))
    mats = omodels.p_t_eigh(q, freqs, bls.unsqueeze(-1) * rates).requires_grad_(True)
    ref = opruning.treelik_discrete_rescaled(tips + [None] * (T - 1), weights, post, mats,
                                             freqs[None], props[:, None, None])
    ref.sum().backward()

    def rel(a, b):
        return float((a.cpu() - b).norm() / b.norm())

    m2 = mats.detach().to(gpu).requires_grad_(True)
    args = (weights.to(gpu), post)
    tail = (freqs[None].to(gpu), props[:, None, None].to(gpu))
    parts = [t.to(gpu) for t in tips] + [None] * (T - 1)
    got = hl.calculate_treelikelihood_discrete(parts, *args, m2, *tail)
    assert rel(got.detach(), ref.detach()) < 1e-12
    got.sum().backward()
    assert rel(m2.grad, mats.grad) < 1e-10
    # without a gradient only the results that wait in memory are stored: the same value
    alone = hl.calculate_treelikelihood_discrete(parts, *args, m2.detach(), *tail)
    assert torch.equal(alone, got.detach())
    # alone or in a batch, one wave or four: the same value
    one = hl.calculate_treelikelihood_discrete(parts, *args, m2.detach()[:1], *tail)
    assert torch.equal(one[0], got.detach()[0])
