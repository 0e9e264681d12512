"""Dense FP32 and split-BF16 post-orders as a walk and by level: the same results to the bit, so that
a sample's result does not depend on the batch that chose between them."""
import numpy as np
import pytest
import torch

from test_walk4_program import _tree

pytestmark = pytest.mark.gpu


# (tree, T, N, K, C, S, dense tips): one sample by level, K as a walk
CASES = [("balanced", 64, 403, 64, 4, 20, False), ("random", 150, 403, 64, 1, 20, True),
         ("balanced", 64, 100, 160, 4, 2, False), ("random", 150, 1000, 32, 3, 8, False),
         ("balanced", 128, 9000, 8, 4, 18, False), ("random", 150, 60, 200, 2, 13, True),
         ("random", 33, 200, 16, 4, 16, False), ("random", 40, 1000, 4, 1, 27, False),
         ("random", 20, 200, 8, 2, 24, True)]


@pytest.mark.parametrize("products", ["fp32", "bf16x3"])
@pytest.mark.parametrize("shape,T,N,K,C,S,dense", CASES)
def test_walk_and_levels_agree_to_the_bit(gpu, shape, T, N, K, C, S, dense, products):
    print(f"case: routes {shape} T={T} N={N} K={K} C={C} S={S} dense={dense} {products}", flush=True)
    from torchtree_amd import _lib
    from torchtree_amd import likelihood as hl

    g = torch.Generator(device=gpu).manual_seed(S * N + T)
    f32, B = torch.float32, 2 * T - 2
    post = _tree(shape, T)
    codes = torch.randint(S + 1, (T, N), generator=g, device=gpu)
    tips = hl.TipData.from_states(list(codes), S, gpu)
    if dense:
        rows = tips.table.to(f32)[codes] * (0.5 + torch.rand(T, N, S, generator=g, device=gpu)) + 0.01
        tips = hl.TipData(_lib.HX_TIPS_DENSE, rows, None, S, N, T)
    mats = torch.rand(1, B, C, S, S, generator=g, device=gpu) + 2 * S * torch.eye(S, device=gpu)
    mats = (mats / mats.sum(-1, keepdim=True)).expand(K, -1, -1, -1, -1).contiguous()
    freqs = torch.full((1, S), 1.0 / S, device=gpu)
    props = torch.full((1, C), 1.0 / C, device=gpu)
    weights = torch.rand(N, generator=g, device=gpu, dtype=torch.float64)
    pr = hl.Pruning(hl.Plan(T, post, 0), tips, weights, products=products)
    code = hl._dtype_code(f32, products)
    few, many = (pr._launches(_lib.HX_GRAD_NONE, S, C, code, k) for k in (1, K))
    assert few > 2 and many == 2, "the two batches take the two routes"
    one = pr.forward(mats[:1].contiguous(), freqs, props)
    all_ = pr.forward(mats, freqs, props)
    for a, b in zip(one[:3], all_[:3]):  # logL, d/dfreqs, d/dprops
        assert torch.equal(a.expand_as(b), b)
    d1 = pr.backward_mats(mats[:1].contiguous(), freqs, props, one[3])
    dk = pr.backward_mats(mats, freqs, props, all_[3])
    assert torch.equal(d1.expand_as(dk), dk)
