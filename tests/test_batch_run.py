"""The groups and launches of a batch call (host build of psl_batch_run.h): groups
of grids that fit the limit together, of about equal size, whatever larger grids
stand between them; and the host shifters when a launch fails: every group of
grids stands at the steps launched for it, in the form of groups and in that of
graphs."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HEADER = os.path.join(os.path.dirname(HERE), "periodicshiftlbm_amd", "csrc", "psl_batch_run.h")


@pytest.fixture(scope="module")
def host():
    out = os.path.join(HERE, "csrc", "_build", "batch_run_host.so")
    src = os.path.join(HERE, "csrc", "batch_run_host.cpp")
    if not os.path.exists(out) or os.path.getmtime(out) < max(os.path.getmtime(src), os.path.getmtime(HEADER)):
        os.makedirs(os.path.dirname(out), exist_ok=True)
        subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-fPIC", "-shared", "-o", out, src], check=True)
    return ctypes.CDLL(out)


@pytest.mark.parametrize("fail", [None, (0, 0), (0, 3), (1, 0), (1, 2), (2, 4)])
def test_group_shifters_follow_the_launched_steps(host, fail):
    groups, steps = 3, 5
    launched, moved = (np.zeros(groups, np.int32) for _ in range(2))
    g, s = fail or (-1, -1)
    rc = host.br_groups(groups, steps, g, s, launched.ctypes.data_as(ctypes.c_void_p),
                        moved.ctypes.data_as(ctypes.c_void_p))
    assert rc == (0 if fail is None else 7)
    assert moved.tolist() == launched.tolist()
    assert moved.tolist() == [steps if fail is None or x < g else s if x == g else 0 for x in range(groups)]


@pytest.mark.parametrize("steps,many,fail,want", [(17, 7, -1, 17), (17, 7, 0, 0), (17, 7, 1, 7), (17, 7, 3, 15),
                                                  (4, 7, -1, 4), (3, 1, 2, 2), (1, 1000, -1, 1), (14, 7, -1, 14)])
def test_graph_shifters_follow_the_launched_steps(host, steps, many, fail, want):
    launched, moved = ctypes.c_int(0), ctypes.c_int(0)
    rc = host.br_graphs(steps, many, fail, ctypes.byref(launched), ctypes.byref(moved))
    assert rc == (0 if fail < 0 else 7)
    assert launched.value == moved.value == want


def _ends(host, sizes, limit, lone=1 << 60):
    b, out = np.array(sizes, np.int64), np.zeros(len(sizes), np.int32)
    n = host.br_ends(len(sizes), b.ctypes.data_as(ctypes.c_void_p), ctypes.c_longlong(limit),
                     ctypes.c_longlong(lone), out.ctypes.data_as(ctypes.c_void_p))
    return out[:n].tolist()


def test_groups_beside_a_larger_grid(host):
    """2 GB ahead of 40 grids of 5 MB: those fill two groups, not one each."""
    assert _ends(host, [2000] + [5] * 40, 192) == [1, 21, 41]
    assert _ends(host, [5] * 40 + [2000], 192) == [20, 40, 41]


@pytest.mark.parametrize("seed", range(20))
def test_groups_fill_the_limit(host, seed):
    """Every grid is in one group; a group of several fits the limit; of two
    neighbouring groups of smaller grids, one is over a quarter of the limit."""
    rng = np.random.default_rng(seed)
    limit = 192
    sizes = np.where(rng.random(60) < 0.1, rng.integers(193, 3000, 60), rng.integers(1, 60, 60)).tolist()
    ends = _ends(host, sizes, limit)
    assert ends[-1] == len(sizes) and all(a < b for a, b in zip(ends, ends[1:]))
    groups = [sizes[a:b] for a, b in zip([0] + ends, ends)]
    for g in groups:
        assert len(g) == 1 or sum(g) <= limit
    for a, b in zip(groups, groups[1:]):
        if max(a + b) <= limit:
            assert max(sum(a), sum(b)) > limit // 4


def test_neighbours_beyond_the_cache_are_one_group(host):
    sizes = [400, 500, 10, 20, 250, 300, 401, 5]
    assert _ends(host, sizes, 192, 350) == [2, 4, 5, 6, 7, 8]
    assert _ends(host, sizes, 192, 249) == [2, 4, 7, 8]
    assert _ends(host, [400, 500, 600], 192, 350) == [3]
