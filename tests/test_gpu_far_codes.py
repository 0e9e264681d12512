"""Four-state FP32 calls whose tip codes reach past 4 GiB: the kernels without 32-bit code offsets."""
import pytest
import torch

from test_walk4_program import _tree

pytestmark = pytest.mark.gpu


def test_codes_past_4_gib(gpu):
    """2100 taxa x 2,050,048 patterns, which repeat 1024: that many times the log-likelihood and
    gradient of the 1024. Tolerances: those of the other FP32 four-state tests."""
    from torchtree_amd import _lib
    from torchtree_amd import likelihood as hl

    T, n, times, S = 2100, 1024, 2002, 4
    assert T * n * times > 1 << 32
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info(gpu)[0] < 130 << 30:
        pytest.skip("needs 130 GiB of device memory")
    g = torch.Generator(device=gpu).manual_seed(1)
    f32 = dict(device=gpu, dtype=torch.float32)
    plan = hl.Plan(T, _tree("random", T), 0)
    site = torch.randint(S, (1, n), generator=g, device=gpu, dtype=torch.uint8)
    other = torch.randint(S + 1, (T, n), generator=g, device=gpu, dtype=torch.uint8)
    codes = torch.where(torch.rand(T, n, generator=g, device=gpu) < 0.3, other, site)
    table = torch.cat((torch.eye(S, **f32), torch.ones(1, S, **f32)))
    mats = torch.rand(1, 2 * T - 2, 1, S, S, generator=g, device=gpu) + 12 * torch.eye(S, device=gpu)
    mats = mats / mats.sum(-1, keepdim=True)
    freqs, props = torch.full((1, S), 1.0 / S, **f32), torch.ones(1, 1, **f32)

    def both(codes):
        N = codes.shape[1]
        tips = hl.TipData(_lib.HX_TIPS_CODES, codes, table, S, N, T)
        pr = hl.Pruning(plan, tips, torch.ones(N, dtype=torch.float64, device=gpu))
        out = pr.forward(mats, freqs, props)
        return out[:3], pr.backward_mats(mats, freqs, props, out[3])

    few, few_d = both(codes)
    print("case: codes past 4 GiB", flush=True)
    many, many_d = both(codes.repeat(1, times))
    torch.cuda.synchronize()

    def rel(a, b):
        return float((a / times - b).norm() / b.norm())

    assert rel(many[0], few[0]) < 1e-6
    for a, b in ((many[1], few[1]), (many[2], few[2]), (many_d, few_d)):
        assert rel(a, b) < 1e-5
    torch.cuda.empty_cache()
