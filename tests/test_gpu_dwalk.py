"""The dense-state FP32 walks where they can go wrong: state counts at the edges of their matrix
shapes, pattern counts at the edges of a tile, every category count, trees that spill and trees that
hold, coded and dense tips, with and without a gradient."""
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


CASES = [("random", 2, 1, 1, 2, False), ("caterpillar", 9, 17, 4, 3, True),
         ("balanced", 16, 15, 2, 5, False), ("random", 33, 16, 3, 16, False),
         ("balanced", 32, 31, 4, 17, False), ("balanced", 64, 50, 4, 20, False),
         ("random", 21, 33, 2, 20, True), ("caterpillar", 12, 48, 1, 20, False),
         ("random", 40, 65, 4, 21, False), ("balanced", 16, 18, 3, 32, True),
         ("random", 30, 100, 4, 32, False)]


# the level kernels of larger state counts: rows of a matrix and of a tile past their ends
LEVEL_CASES = [("random", 9, 1, 1, 33, False), ("balanced", 16, 17, 4, 49, False),
               ("random", 12, 33, 2, 61, True), ("caterpillar", 7, 150, 3, 61, False),
               ("random", 20, 140, 4, 64, False)]


@pytest.mark.parametrize("shape,T,N,C,S,dense", CASES + LEVEL_CASES)
def test_dense_walks(gpu, shape, T, N, C, S, dense):
    """Tolerances: those of the other FP32 tests (logL 1e-6, gradients 1e-5 norm-wise)."""
    print(f"case: dense FP32 passes {shape} T={T} N={N} C={C} S={S} dense={dense}", flush=True)
    from torchtree_amd import likelihood as hl
    from torchtree_amd.serving import ResidentJob

    rng = np.random.default_rng(1000 * S + T * N)
    post, K, B = _tree(shape, T), 3, 2 * T - 2
    # patterns with a signal: a state of the site, in some tips another or an unknown one
    codes = (rng.integers(0, S, size=(1, N)) + (rng.random((T, N)) < 0.3) * rng.integers(0, S, (T, N))) % S
    codes = np.where(rng.random((T, N)) < 0.05, S, codes)
    table = np.vstack((np.eye(S), np.ones((1, S))))
    tips = [torch.tensor(table[codes[t]].T.copy()) for t in range(T)]
    if dense:
        tips = [t * torch.tensor(rng.uniform(0.2, 1.0, t.shape)) + 0.01 for t in tips]
    weights = torch.tensor(rng.integers(1, 5, N).astype(float))
    freqs = torch.tensor(rng.dirichlet(np.full(S, 10.0)))
    q = omodels.q_from_exchangeabilities(torch.tensor(rng.gamma(2.0, 2.0, S * (S - 1) // 2)), freqs)
    rates = torch.linspace(0.3, 2.0, C, dtype=F64) if C > 1 else torch.ones(1, dtype=F64)
    props = torch.full((C,), 1.0 / C, dtype=F64)
    bls = torch.tensor(rng.exponential(0.1, (K, B)), requires_grad=True)
    mats = omodels.p_t_eigh(q, freqs, bls.unsqueeze(-1) * rates)
    mats.retain_grad()
    ref = opruning.treelik_discrete_rescaled(tips + [None] * (T - 1), weights, post, mats,
                                             freqs[None], props[:, None, None])
    ref.sum().backward()

    def rel(a, b):
        return float((a.double().cpu() - b).norm() / b.norm())

    f32 = dict(device=gpu, dtype=torch.float32)
    m2 = mats.detach().to(**f32).requires_grad_(True)
    args = (weights.to(gpu), post)
    tail = (freqs[None].to(**f32), props[:, None, None].to(**f32))
    parts = [t.to(gpu) for t in tips] + [None] * (T - 1)
    got = hl.calculate_treelikelihood_discrete(parts, *args, m2, *tail)
    assert rel(got.detach(), ref.detach()) < 1e-6
    got.sum().backward()
    assert rel(m2.grad, mats.grad) < 1e-5
    # without a gradient only the results that wait in memory are stored: the same value
    alone = hl.calculate_treelikelihood_discrete(parts, *args, m2.detach(), *tail)
    assert torch.equal(alone, got.detach())
    if not dense:
        # d logL / d tau: the resident job's form
        job = ResidentJob("dwalk", post, codes.astype(np.uint8), table, weights.numpy(),
                          q / -(torch.diagonal(q) * freqs).sum(), freqs.numpy(), rates.numpy(),
                          props.numpy(), dtype=torch.float32)
        ll = torch.empty(K, dtype=F64, device=gpu)
        db = torch.empty(K, B, dtype=F64, device=gpu)
        ws = torch.full((job.workspace_bytes(K),), 255, dtype=torch.uint8, device=gpu)
        job.eval(bls.detach().to(gpu), ll, db, ws, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert rel(ll, ref.detach().reshape(-1)) < 1e-6
        assert rel(db, bls.grad) < 1e-5
