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
    L.cols_pay.restype, L.cols_pay.argtypes = i, [i64, i64, i64, i64, i, i, C.POINTER(C.c_double)]
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


@pytest.mark.parametrize("M,N,K,tile", [(2176, 512, 6144, (128, 128)), (343, 3072, 6144, (128, 128)),
                                        (700, 1536, 6144, (128, 128)), (867, 1152, 4544, (64, 64))])
def test_long_products_on_few_tiles(host, M, N, K, tile):
    """half a chip of 64 x 128 tiles walking a long K takes longer than split 128 x 128 or 64 x 64 ones"""
    assert plan(host, M, N, K)[:2] == tile


# the forward products of a block of width d: (outputs, inputs, paired SwiGLU, heads prepared)
def block_products(d):
    return {"qkv": (5 * d, d, 0, 1), "out": (d, d, 0, 0), "cross.q": (2 * d, d, 0, 1), "cross.out": (d, d, 0, 0),
            "ff.proj": (8 * d, d, 1, 0), "ff.out": (d, 4 * d, 0, 0)}


def test_rank_columns_ride_where_they_cost_less_than_a_product(host):
    """the benchmark's 2176 rows of width 1536: only the QKV product, which the columns would cost a round
    of 128 x 256 tiles, leaves its rank product to launches of its own"""
    own = C.c_double()
    ride = {n: host.cols_pay(2176, N, K, 32, sw, h, C.byref(own)) for n, (N, K, sw, h) in block_products(1536).items()}
    assert ride == {"qkv": 0, "out": 1, "cross.q": 1, "cross.out": 1, "ff.proj": 1, "ff.out": 1}
    for M, N, K in sizes():
        if N <= 64:
            continue
        ride = host.cols_pay(M, N, K, 16, 0, 0, C.byref(own))
        assert ride == (plan(host, M, N + 16, K)[4] <= plan(host, M, N, K)[4] + own.value)
