"""The tile and split choice of bf16 products (csrc/gemm_plan.h), which is host arithmetic: compiled
with g++ and checked without a GPU over the sizes the entry points take."""
import ctypes as C
import os
import random
import subprocess

import pytest

from conftest import PKG, ROOT

CUS, LDS = 256, 160 * 1024


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("gemm_plan") / "libgemm_plan.so")
    cmd = ["g++", "-std=c++17", "-O2", "-fPIC", "-shared", "-Wall", "-Wextra", "-Werror", "-I", os.path.join(PKG, "csrc"),
           os.path.join(ROOT, "tests", "host", "gemm_plan_shim.cpp"), "-o", out]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    L = C.CDLL(out)
    i64, i = C.c_int64, C.c_int
    L.plan.restype, L.plan.argtypes = C.c_double, [i64, i64, i64, i, i, i, i, C.POINTER(i)]
    return L


def plan(host, M, N, K, split=1, big=1, swiglu=0, heads=0):
    """(tile rows, tile columns, LDS stages, splits, us)"""
    out = (C.c_int * 4)()
    us = host.plan(M, N, K, split, big, swiglu, heads, out)
    return (*out, us)


def sizes():
    """rows, columns and K of products: every small row count, then all ranges at random"""
    for M in (1, 2, 3, 8, 10, 16, 31, 32, 33, 64, 100):
        for N in range(128, 9217, 448):
            for K in range(64, 9601, 448):
                yield M, N, K
    r = random.Random(5)
    for _ in range(4000):
        yield int(2 ** r.uniform(0, 13)), 8 * r.randint(9, 2100), 64 * r.randint(1, 200)
    # refused when the plan counted on two 32 x 128 workgroups to a CU
    yield from ((1, 3072, 3072), (3, 4608, 2304), (3, 2304, 6144), (2, 4096, 2304), (10, 2176, 9216), (32, 16448, 9600))


def test_splits_fit_the_resident_workgroups(host):
    """splits x tiles stays within the workgroups that the tile's LDS lets the chip hold: the launcher
    refuses any other plan (its partial sums are sized by that bound)"""
    for M, N, K in sizes():
        rows, cols, stages, s, _ = plan(host, M, N, K)
        slots = CUS * max(1, LDS // (stages * (rows + cols) * 128 + 64))
        tiles = -(-M // rows) * -(-N // cols)
        assert s == 1 or s * tiles <= slots, (M, N, K, rows, cols, s)
        assert 1 <= s <= max(1, K // 64 // 4)
        assert plan(host, M, N, K, split=0)[3] == 1
