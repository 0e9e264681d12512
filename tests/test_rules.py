"""The dispatch rules of csrc/layout.hpp, compiled with g++ from the library's own header."""
import shutil
import subprocess

import pytest

from torchtree_amd.build import CSRC

HERE = __import__("pathlib").Path(__file__).parent


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    out = tmp_path_factory.mktemp("rules") / "rules_dump"
    subprocess.run(["g++", "-O1", "-std=c++17", f"-I{CSRC}", f"-I{HERE.parent / 'include'}",
                    str(HERE / "native" / "rules_dump.cpp"), "-o", str(out)], check=True)

    def run(lines):
        text = "\n".join(" ".join(map(str, ln)) for ln in lines)
        r = subprocess.run([str(out)], input=text, capture_output=True, text=True, check=True)
        return [int(x) for x in r.stdout.split()]

    return run


def test_post_level_tiles_cover_every_shape(ask):
    """Always 1 .. min(ntiles, 64) tiles, whatever the shape."""
    grid = [("tiles", S, nt, C, K, w, f) for S in (2, 16, 17, 20, 21, 32, 33, 61, 64)
            for nt in (1, 2, 7, 63, 64, 65, 1250, 200000) for C in (1, 2, 3, 4) for K in (1, 8, 1024)
            for w in (1, 2, 512) for f in (0, 1)]
    got = ask(grid)
    assert len(got) == len(grid)
    for q, t in zip(grid, got):
        assert 1 <= t <= min(q[2], 64), q


@pytest.mark.parametrize("S", [2, 8, 16, 20])
@pytest.mark.parametrize("f64", [0, 1])
def test_post_level_tiles_leave_blocks_to_share_a_cu(ask, S, f64):
    """Up to 20 states several blocks share a CU: a level that could give every CU eight blocks of
    one tile gives it at least four."""
    for nt, K, w in ((188, 8, 13), (188, 1, 64), (25, 8, 64), (1250, 1, 10)):
        t, = ask([("tiles", S, nt, 4, K, w, f64)])
        assert (nt + t - 1) // t * K * w >= 4 * 256, (nt, K, w, t)


@pytest.mark.parametrize("S", [2, 8, 16, 18, 20, 27, 32])
@pytest.mark.parametrize("C", [1, 2, 3, 4])
def test_dense_walk_only_where_its_chain_is_hidden(ask, S, C):
    """A walk's time at few patterns is the chain of all its nodes, a level's a launch: few patterns
    on a bushy tree go by level, a caterpillar walks; past 32 states there is no walk."""
    assert ask([("dwalk", S, C, 127, 7, 1, 1), ("dwalk", S, C, 349, 18, 4, 1),
                ("dwalk", S, C, 199, 199, 1, 1), ("dwalk", 33, C, 199, 199, 1, 1)]) == [0, 0, 1, 0]


def test_tau_chunks_grow_with_the_patterns(ask):
    """Short chunks where there are few blocks, longer ones before their set-ups outweigh that, never
    longer than the d/dP chunks'."""
    assert ask([("tau", 77, 4, 9), ("tau", 188, 4, 9), ("tau", 500, 4, 9), ("tau", 1000, 4, 8),
                ("tau", 5000, 1, 40), ("tau", 188, 1, 9), ("tau", 500, 1, 9), ("tau", 7, 4, 7),
                ("tau", 1, 1, 1)]) == [5, 6, 8, 8, 40, 5, 6, 5, 1]


@pytest.mark.parametrize("S", [33, 61, 64])
def test_post_level_tiles_of_one_category_stay_short(ask, S):
    """One category at 33 states and more: at most 10 tiles a block, whatever the launch holds."""
    grid = [("tiles", S, nt, 1, K, w, f) for nt in (1, 7, 100, 1250, 6250, 65536) for K in (1, 8, 32)
            for w in (1, 9, 64) for f in (0, 1)]
    for q, t in zip(grid, ask(grid)):
        assert 1 <= t <= min(q[2], 10), q


def test_rows_as_operands_where_they_are_short_or_used_once(ask):
    """Past 20 states rows, but with coded tips at 3 categories; one tile's post-order of 20 and fewer never; below 16 states and with
    split products of 17 and 19 never."""
    for S in range(2, 65):
        for C in (1, 2, 3, 4):
            for split in (0, 1):
                pre, one, many = ask([("nat", S, C, split, 0, 1, 1), ("nat", S, C, split, 1, 1, 1),
                                      ("nat", S, C, split, 1, 400, 1)])
                assert pre == many
                coded = ask([("nat", S, C, split, 0, 1, 0), ("nat", S, C, split, 1, 400, 0)])
                assert coded == [pre, many and not (20 < S < 32 and C == 3 and not split)]
                if S > 20:
                    assert one == many == 1
                else:
                    assert one == 0 and not (many and (S < 16 or split and S in (17, 19)))


@pytest.mark.parametrize("S,C", [(8, 4), (17, 2), (18, 1), (18, 2), (19, 4), (24, 3), (32, 2)])
def test_dense_tips_of_many_patterns_go_by_level(ask, S, C):
    """Rows of dense tips come word by word in the walk: a large batch on a balanced tree goes by level,
    which the same call with 20 states does not."""
    assert ask([("route", S, C, 199, 8, 625, 16, 1, f) for f in (0, 1)]) == [0, 0]
    assert ask([("route", 20, C, 199, 8, 625, 16, 1, f) for f in (0, 1)]) == [1, 1]
