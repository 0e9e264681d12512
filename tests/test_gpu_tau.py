"""hx_loglik_grad_tau through the C entry points: coded and dense tips, both precisions, every
category count, and the contraction with dP/dtau where its rows cancel."""
import numpy as np
import pytest
import torch

from oracle import pruning as opruning
from test_walk4_program import _tree

pytestmark = pytest.mark.gpu
F64 = torch.float64


def _call(gpu, post, tips, table, weights, mats, mats_dt, dtype, first=2):
    """(logL [K], d/dtau [K, B, C]) of hx_loglik and hx_loglik_grad_tau; tips [T, N] codes with a
    table, or [T, N, S]. first: the gradient mode whose workspace size hx_loglik is told."""
    from torchtree_amd import _lib
    from torchtree_amd.likelihood import Plan, _dtype_code

    lib = _lib.load()
    K, B, C, S, _ = mats.shape
    T, N = tips.shape[:2]
    plan, code = Plan(T, post, 0), _dtype_code(dtype, "fp32")
    dev = dict(device=gpu, dtype=dtype)
    mats, mats_dt = mats.to(**dev).contiguous(), mats_dt.to(**dev).contiguous()
    freqs, props = torch.full((1, S), 1.0 / S, **dev), torch.full((1, C), 1.0 / C, **dev)
    dense = table is None
    tips = (tips.to(**dev) if dense else tips.to(gpu, torch.uint8)).contiguous()
    table = None if dense else table.to(**dev).contiguous()
    weights = weights.to(gpu)
    nb = plan.workspace_bytes(S, N, C, K, code, _lib.HX_GRAD_TAU)
    ws = torch.full((nb,), 255, dtype=torch.uint8, device=gpu)
    ll = torch.empty(K, dtype=F64, device=gpu)
    dt = torch.empty(K, B, C, dtype=F64, device=gpu)
    head = (plan.handle, S, N, C, K, code, int(dense), tips.data_ptr(), _lib.ptr(table),
            0 if dense else table.shape[0], weights.data_ptr(), mats.data_ptr())
    tail = (freqs.data_ptr(), 0, props.data_ptr(), 0, ws.data_ptr(), nb)
    st = _lib.stream_handle(gpu)
    small = plan.workspace_bytes(S, N, C, K, code, first)
    _lib.check(lib.hx_loglik(*head, *tail[:-1], small, ll.data_ptr(), 0, 0, st))
    _lib.check(lib.hx_loglik_grad_tau(*head, mats_dt.data_ptr(), *tail, dt.data_ptr(), st))
    torch.cuda.synchronize()
    return ll.cpu(), dt.cpu()


def _oracle(post, rows, weights, mats, mats_dt):
    """The same in 64 bits: rows [T, N, S]."""
    K, B, C, S, _ = mats.shape
    m = mats.double().requires_grad_(True)
    ref = opruning.treelik_discrete_rescaled(
        [r.T.contiguous() for r in rows.double()] + [None] * (rows.shape[0] - 1), weights, post, m,
        torch.full((1, S), 1.0 / S, dtype=F64), torch.full((C, 1, 1), 1.0 / C, dtype=F64))
    ref.sum().backward()
    return ref.detach().reshape(-1), (m.grad * mats_dt.double()).sum((-1, -2))


CASES = [("random", 9, 70, 3, 4), ("balanced", 16, 64, 4, 4), ("caterpillar", 12, 130, 1, 4),
         ("random", 30, 257, 2, 4), ("random", 20, 33, 4, 20), ("balanced", 8, 40, 2, 61)]


@pytest.mark.parametrize("dtype", [torch.float32, F64])
@pytest.mark.parametrize("dense", [False, True])
@pytest.mark.parametrize("shape,T,N,C,S", CASES)
def test_grad_tau(gpu, shape, T, N, C, S, dense, dtype):
    """Tolerances: those of the other tests of these passes (FP32 logL 1e-6, gradient 1e-5
    norm-wise; FP64 1e-10)."""
    print(f"case: grad_tau {shape} T={T} N={N} C={C} S={S} dense={dense} {dtype}", flush=True)
    rng = np.random.default_rng(T * N + S)
    post, K, B = _tree(shape, T), 2, 2 * T - 2
    codes = (rng.integers(0, S, (1, N)) + (rng.random((T, N)) < 0.3) * rng.integers(0, S, (T, N))) % S
    codes = np.where(rng.random((T, N)) < 0.05, S, codes)
    table = torch.tensor(np.vstack((np.eye(S), np.ones((1, S)))))
    rows = table[torch.tensor(codes)]
    if dense:
        rows = rows * torch.tensor(rng.uniform(0.2, 1.0, rows.shape)) + 0.01
    # (inputs at the call's precision, so that both sides see the same ones)
    near = lambda x: torch.tensor(x).to(dtype).double()  # noqa: E731
    rows = rows.to(dtype).double()
    mats = rng.uniform(0.1, 1.0, (K, B, C, S, S)) + 3 * S * np.eye(S)
    mats = near(mats / mats.sum(-1, keepdims=True))
    mats_dt = near(rng.standard_normal((K, B, C, S, S)))
    weights = torch.tensor(rng.integers(1, 5, N).astype(float))
    ll, dt = _call(gpu, post, rows if dense else torch.tensor(codes), None if dense else table,
                   weights, mats, mats_dt, dtype)
    ref_ll, ref_dt = _oracle(post, rows, weights, mats, mats_dt)
    f32 = dtype == torch.float32
    assert float((ll - ref_ll).norm() / ref_ll.norm()) < (1e-6 if f32 else 1e-10)
    assert float((dt - ref_dt).norm() / ref_dt.norm()) < (1e-5 if f32 else 1e-10)


@pytest.mark.parametrize("C", [1, 2, 3, 4])
def test_grad_tau_contracts_in_64_bits(gpu, C):
    """Rows 2^24, 1, -2^24, 0 of dP/dtau against equal partials: 1 in 64 bits, where 32 bits round
    2^24 + 1 and leave 0. FP32 up to the contraction: the ratio of adjoint and likelihood, to 1e-5."""
    T, N, K, B = 6, 70, 2, 10
    post = _tree("random", T)
    rng = np.random.default_rng(C)
    mats = rng.uniform(0.1, 1.0, (K, B, C, 4, 4)) + 4 * np.eye(4)
    mats = torch.tensor(mats / mats.sum(-1, keepdims=True)).float().double()
    mats_dt = torch.tensor([2.0**24, 1.0, -(2.0**24), 0.0]).expand(K, B, C, 4, 4)
    weights = torch.tensor(rng.integers(1, 5, N).astype(float))
    table = torch.cat((torch.eye(4), torch.ones(1, 4)))
    codes = torch.full((T, N), 4)
    _, dt = _call(gpu, post, codes, table, weights, mats, mats_dt, torch.float32)
    _, ref = _oracle(post, table[codes], weights, mats, mats_dt)
    tips = slice(0, T)  # branches of tips, whose partials are ones exactly
    assert torch.allclose(ref[:, tips].sum(-1), weights.sum().expand(K, T), rtol=1e-5)
    assert float((dt[:, tips] - ref[:, tips]).abs().max() / ref[:, tips].abs().max()) < 1e-5


@pytest.mark.parametrize("dtype", [torch.float32, F64])
@pytest.mark.parametrize("shape,T,N,C,S", [("balanced", 16, 64, 4, 4), ("caterpillar", 20, 33, 4, 20)])
def test_partials_are_kept_whatever_size_is_told(gpu, shape, T, N, C, S, dtype):
    """A caller with one buffer for both calls may tell hx_loglik the size without a gradient: its
    partials are there all the same."""
    from torchtree_amd import _lib

    rng = np.random.default_rng(T)
    post, K, B = _tree(shape, T), 2, 2 * T - 2
    mats = torch.tensor(rng.uniform(0.1, 1.0, (K, B, C, S, S)) + S * np.eye(S))
    mats = mats / mats.sum(-1, keepdim=True)
    mats_dt = torch.tensor(rng.standard_normal((K, B, C, S, S)))
    weights = torch.ones(N, dtype=F64)
    args = (post, torch.tensor(rng.integers(0, S, (T, N))), torch.eye(S), weights, mats, mats_dt, dtype)
    told = _call(gpu, *args, first=_lib.HX_GRAD_NONE)
    for a, b in zip(told, _call(gpu, *args)):
        assert torch.equal(a, b)
