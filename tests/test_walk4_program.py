"""The programs of the four-state FP32 walks (csrc/walk.hpp, build_post4 and build_pre4).

Compiled with g++ from the library's own header and executed here in FP64 numpy as the kernels
execute them: results that wait are held in registers or read back from memory, dropped cherries
are never stored and are rebuilt from their tips, adjoints are held, pushed into their partial's
place or continued. Log-likelihood and d/dP equal the oracle's on every kind of tree.
"""
import math
import shutil
import subprocess

import numpy as np
import pytest

from torchtree_amd import synthetic
from torchtree_amd.build import CSRC

HERE = __import__("pathlib").Path(__file__).parent


@pytest.fixture(scope="module")
def walk4_bin(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    out = tmp_path_factory.mktemp("walk4") / "walk4_dump"
    subprocess.run(["g++", "-O1", "-std=c++17", f"-I{CSRC}",
                    str(HERE / "native" / "walk4_dump.cpp"), "-o", str(out)], check=True)
    return out


def _programs(walk4_bin, T, post):
    inp = f"{T}\n" + "\n".join(f"{v} {a} {b}" for v, a, b in post) + "\n"
    r = subprocess.run([str(walk4_bin)], input=inp, capture_output=True, text=True, check=True)
    lines = [tuple(int(x) for x in ln.split()) for ln in r.stdout.splitlines() if ln.strip()]
    (slots, need), rest = lines[0], lines[1:]
    return slots, need, rest[: T - 1], rest[T - 1:]


def _tree(shape, T):
    if shape == "random":
        topo = synthetic.random_topology(T, np.random.default_rng(T))
        return [tuple(int(x) for x in r) for r in topo.postorder]
    if shape == "caterpillar":
        post, prev = [], 0
        for i, t in enumerate(range(1, T)):
            post.append((T + i, t, prev) if i % 2 else (T + i, prev, t))
            prev = T + i
        return post
    level, post, nxt = list(range(T)), [], T
    while len(level) > 1:
        new = []
        for i in range(0, len(level) - 1, 2):
            post.append((nxt, level[i], level[i + 1]))
            new.append(nxt)
            nxt += 1
        level = new + (level[-1:] if len(level) % 2 else [])
    return post


def _post(T, prog, slots, P, tips):
    """Partials left in memory and the root's, with the kernel's registers and stack."""
    mv = lambda b, x: np.einsum("cij,cjn->cin", P[b], x)  # noqa: E731
    C = P.shape[1]
    tip = lambda t: np.broadcast_to(tips[t], (C,) + tips[t].shape)  # noqa: E731
    mem, stack, y, held = {}, [None] * slots, None, None
    for i, (c1, c2, v, m) in enumerate(prog):
        kind = m & 3
        if m & 4:
            held = y
        assert (c1 < T) == (kind <= 1) and (c2 < T) == (kind == 0)
        x2 = tip(c2) if kind == 0 else y
        if kind <= 1:
            x1 = tip(c1)
        elif kind == 2:
            x1, held = held, None
        else:
            assert stack[(m >> 8) & 0xFF] == c1
            x1 = mem[c1]
        if kind:
            assert prog[i - 1][2] == c2  # the previous result
        y = mv(c1, x1) * mv(c2, x2)
        if m & 16:
            assert not m & 8
            stack[(m >> 16) & 0xFF] = v
        if not m & 8:
            mem[v] = y
    return mem, y


def _pre(T, prog, P, tips, mem, freqs, props, weights):
    mv = lambda b, x: np.einsum("cij,cjn->cin", P[b], x)  # noqa: E731
    C, N = P.shape[1], tips[0].shape[-1]
    tip = lambda t: np.broadcast_to(tips[t], (C,) + tips[t].shape)  # noqa: E731
    rows = {v: ("L", x) for v, x in mem.items()}
    grad, U, held = np.zeros_like(P), None, None
    for p, c1, c2, m, *g in prog:
        src = m & 3
        if src == 0:
            U = np.broadcast_to(freqs[:, None], (C, 4, N))
        elif src == 2:
            kind, U = rows[p]
            assert kind == "U"
        elif src == 3:
            U, held = held, None
        assert U is not None
        L = []
        for h, ch in enumerate((c1, c2)):
            kind = (m >> (2 + 2 * h)) & 3
            if kind == 0:
                assert ch < T
                L.append(tip(ch))
            elif kind == 1:
                assert ch not in mem  # never stored
                a, b = g[2 * h: 2 * h + 2]
                L.append(mv(a, tip(a)) * mv(b, tip(b)))
            else:
                what, x = rows[ch]
                assert what == "L"
                L.append(x)
        m1, m2 = mv(c1, L[0]), mv(c2, L[1])
        ut = [U * m2, U * m1]
        lik = np.einsum("c,cin->n", props, ut[0] * m1)
        for h, ch in enumerate((c1, c2)):
            grad[ch] = np.einsum("n,c,cin,cjn->cij", weights / lik, props, ut[h], L[h])
        adjoint = lambda h, ch: np.einsum("cij,cin->cjn", P[ch], ut[h])  # noqa: E731
        push = (m >> 6) & 3
        if push == 1:
            rows[c1] = ("U", adjoint(0, c1))
        elif push == 2:
            assert held is None
            held = adjoint(0, c1)
        U = adjoint(1, c2) if m & 256 else None
    assert held is None
    return grad


@pytest.mark.parametrize("shape,T", [("random", 2), ("random", 3), ("random", 6), ("random", 41),
                                     ("random", 200), ("caterpillar", 3), ("caterpillar", 30),
                                     ("balanced", 4), ("balanced", 8), ("balanced", 64),
                                     ("balanced", 100)])
def test_walk4_programs_match_oracle(walk4_bin, shape, T):
    import torch

    from oracle import pruning as orc

    post = _tree(shape, T)
    slots, need, post4, pre4 = _programs(walk4_bin, T, post)
    assert len(post4) == len(pre4) == T - 1
    assert [e[2] for e in post4][-1] == post[-1][0]
    assert slots <= max(0, need - 1)
    if shape == "caterpillar" or T <= 4:
        assert slots == 0  # one held result is enough
    if shape == "balanced" and T & (T - 1) == 0:
        assert slots == max(0, int(math.log2(T)) - 2)
    cherries = sum(a < T and b < T for v, a, b in post[:-1])
    assert sum(bool(e[3] & 8) for e in post4) == cherries

    rng = np.random.default_rng(T)
    C, N, B = 3, 7, 2 * T - 2
    P = rng.dirichlet(np.ones(4), size=(B, C, 4))
    freqs, props = rng.dirichlet(np.ones(4)), rng.dirichlet(np.ones(C))
    tips = rng.uniform(0.05, 1.0, size=(T, 4, N))
    weights = rng.integers(1, 5, size=N).astype(np.float64)
    mem, root = _post(T, post4, slots, P, tips)
    lik = np.einsum("c,i,cin->n", props, freqs, root)
    grad = _pre(T, pre4, P, tips, mem, freqs, props, weights)

    tm = torch.tensor(P, requires_grad=True)
    parts = [torch.tensor(tips[t]) for t in range(T)] + [None] * (T - 1)
    ll = orc.treelik_discrete(parts, torch.tensor(weights), post, tm, torch.tensor(freqs)[None],
                              torch.tensor(props)[:, None, None])
    ll.sum().backward()
    np.testing.assert_allclose((weights * np.log(lik)).sum(), ll.item(), rtol=1e-12)
    np.testing.assert_allclose(grad, tm.grad.numpy(), rtol=1e-10, atol=1e-12)
