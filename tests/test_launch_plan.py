"""The launch plans' host arithmetic (csrc/chunk_plan.h), compiled here."""

import ctypes
import os
import random
import subprocess

import pytest

import ludwig_amd


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text("""
#include "chunk_plan.h"
extern "C" int count(int nx, long long ncol, int slots) { return ldw::chunk_count(nx, ncol, slots); }
extern "C" long long cost(int nx, long long ncol, int slots, int n) { return ldw::chunk_cost(nx, ncol, slots, n); }
""")
    csrc = os.path.join(os.path.dirname(ludwig_amd.__file__), "csrc")
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", csrc, "-o", str(d / "plan.so"), str(d / "plan.cpp")],
                   check=True)
    so = ctypes.CDLL(str(d / "plan.so"))
    so.cost.restype = ctypes.c_longlong
    return lambda nx, ncol, slots: so.count(nx, ctypes.c_longlong(ncol), slots), \
        lambda nx, ncol, slots, n: so.cost(nx, ctypes.c_longlong(ncol), slots, n)


def test_chunks_are_the_cheapest(plan):
    count, cost = plan
    rng = random.Random(1)
    cases = [(1, 1, 1024), (1, 5000, 1024), (64, 648, 1280), (256, 1280, 1280), (256, 1281, 1280), (3, 2, 256)]
    cases += [(rng.randint(1, 300), rng.choice([rng.randint(1, 60), rng.randint(1, 6000)]),
               rng.choice([256, 768, 1024, 1280, 2560])) for _ in range(300)]
    for nx, ncol, slots in cases:
        n = count(nx, ncol, slots)
        assert 1 <= n <= nx
        least = min(cost(nx, ncol, slots, k) for k in range(1, nx + 1))
        assert cost(nx, ncol, slots, n) == least, (nx, ncol, slots, n)


def test_no_gap_between_half_and_all_of_the_slots(plan):
    # columns that fill more than half of the slots once: marching through all
    # planes in one round leaves the rest idle, chunks in several rounds do not
    count, cost = plan
    for ncol in (641, 700, 900):
        assert count(288, ncol, 1280) > 1
        assert cost(288, ncol, 1280, count(288, ncol, 1280)) < 0.8 * (288 + 3)
