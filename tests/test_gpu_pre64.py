"""The four-state FP64 pre-order walk and the sum of its statistics where they can go wrong: a tile's
quarters, tile counts around the sum's parts and its unrolled turn, trees that push and trees that
only go on, every category count."""
import numpy as np
import pytest
import torch

from oracle import models as omodels
from oracle import pruning as opruning
from test_walk4_program import _tree

pytestmark = pytest.mark.gpu
F64 = torch.float64

# parts of the sum: 8 (4 categories), 10, 16, 32; eight of them are one turn
CASES = [("random", 2, 1, 4, 2), ("caterpillar", 7, 16, 1, 1), ("balanced", 16, 49, 2, 3), ("random", 40, 64, 3, 2),
         ("random", 21, 64 * 8 + 1, 4, 1), ("balanced", 8, 64 * 57, 4, 2), ("random", 9, 64 * 64 - 5, 4, 1),
         ("random", 9, 64 * 73 + 1, 3, 1), ("random", 5, 64 * 130, 2, 1), ("balanced", 8, 64 * 260 + 33, 1, 1),
         ("random", 60, 100, 4, 2), ("random", 200, 64 * 132, 4, 1), ("caterpillar", 120, 100, 2, 2),
         # by tree level: few patterns on a large tree
         ("random", 300, 90, 4, 1), ("balanced", 256, 130, 1, 2)]


@pytest.mark.parametrize("shape,T,N,C,K", CASES)
def test_pre_walk64(shape, T, N, C, K):
    """Both gradients against the oracle to 1e-10 norm-wise, as the other FP64 tests; a sample's
    gradient alone or in a batch is the same bits."""
    print(f"case: FP64 pre-order walk {shape} T={T} N={N} C={C} K={K}", flush=True)
    from torchtree_amd import likelihood as hl
    from torchtree_amd.serving import ResidentJob

    gpu = torch.device("cuda", 0)
    rng = np.random.default_rng(7 * T * N + C)
    post, B = _tree(shape, T), 2 * T - 2
    codes = (rng.integers(0, 4, size=(1, N)) + (rng.random((T, N)) < 0.3) * rng.integers(0, 4, (T, N))) % 4
    codes = np.where(rng.random((T, N)) < 0.05, 4, codes)
    table = np.vstack((np.eye(4), np.ones((1, 4))))
    tips = [torch.tensor(table[codes[t]].T.copy()) for t in range(T)]
    weights = torch.tensor(rng.integers(1, 5, N).astype(float))
    freqs = torch.tensor(rng.dirichlet(np.full(4, 10.0)))
    q = omodels.gtr_q(torch.tensor(rng.gamma(2.0, 2.0, 6)), freqs)
    rates = torch.linspace(0.3, 2.0, C, dtype=F64) if C > 1 else torch.ones(1, dtype=F64)
    props = torch.tensor(rng.dirichlet(np.full(C, 5.0)))
    bls = torch.tensor(rng.exponential(0.1, (K, B)), requires_grad=True)
    mats = omodels.p_t_eigh(q, freqs, bls.unsqueeze(-1) * rates)
    mats.retain_grad()
    ref = opruning.treelik_discrete_rescaled(tips + [None] * (T - 1), weights, post, mats,
                                             freqs[None], props[:, None, None])
    ref.sum().backward()

    def rel(a, b):
        return float((a.cpu() - b).norm() / b.norm())

    def dmats(m):
        m = m.detach().to(gpu).requires_grad_(True)
        hl.calculate_treelikelihood_discrete([t.to(gpu) for t in tips] + [None] * (T - 1), weights.to(gpu), post, m,
                                             freqs[None].to(gpu), props[:, None, None].to(gpu)).sum().backward()
        return m.grad

    got = dmats(mats)
    assert rel(got, mats.grad) < 1e-10
    assert torch.equal(dmats(mats[-1:])[0], got[-1])
    # d logL / d tau: the resident job's form
    job = ResidentJob("pre64", post, codes.astype(np.uint8), table, weights.numpy(),
                      q / -(torch.diagonal(q) * freqs).sum(), freqs.numpy(), rates.numpy(), props.numpy(), dtype=F64)
    ll = torch.empty(K, dtype=F64, device=gpu)
    db = torch.empty(K, B, dtype=F64, device=gpu)
    ws = torch.full((job.workspace_bytes(K),), 255, dtype=torch.uint8, device=gpu)
    job.eval(bls.detach().to(gpu), ll, db, ws, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert rel(ll, ref.detach().reshape(-1)) < 1e-12
    assert rel(db, bls.grad) < 1e-10
