"""What a batch call leaves in the host shifters when a launch fails (host build
of psl_batch_run.h): every group of grids stands at the steps launched for it,
in the form of groups and in that of graphs."""
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
