"""The column splits of the merged adapter refresh (csrc/refresh_plan.h), which are host arithmetic:
compiled with g++ and checked without a GPU."""
import ctypes as C
import os
import random
import subprocess

import pytest

from conftest import PKG, ROOT

COUNTERS = 8192   # arrival counters of a stream


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("refresh_plan") / "librefresh_plan.so")
    cmd = ["g++", "-std=c++17", "-O2", "-fPIC", "-shared", "-Wall", "-Wextra", "-Werror", "-I", os.path.join(PKG, "csrc"),
           os.path.join(ROOT, "tests", "host", "refresh_plan_shim.cpp"), "-o", out]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    L = C.CDLL(out)
    L.refresh.restype = C.c_int64
    L.refresh.argtypes = [C.POINTER(C.c_int64), C.c_int, C.c_int, C.c_int64, C.POINTER(C.c_int)]
    return L


def refresh(host, shapes, dora, counters=COUNTERS):
    flat = (C.c_int64 * (2 * len(shapes)))(*[v for s in shapes for v in s])
    splits = (C.c_int * len(shapes))()
    return host.refresh(flat, len(shapes), dora, counters, splits), list(splits)


def block(dim, inner):
    return [(dim, 5 * dim), (dim, dim), (dim, 2 * dim), (dim, 3 * dim), (dim, dim), (dim, 2 * inner), (inner, dim)]


def test_splits_of_known_refreshes(host):
    assert refresh(host, [(1536, 6144)], 1)[1] == [6]                     # one linear: 4 chunks a workgroup
    assert set(refresh(host, block(1536, 6144) * 24, 1)[1]) == {1}        # the rows alone fill the chip
    assert refresh(host, [(1536, 6144)], 1, counters=0)[1] == [1]         # no counters on the stream
    assert refresh(host, [(1536, 6144)], 0, counters=0)[1] == [6]         # lora needs none


def test_dora_falls_back_past_the_arrival_counters(host):
    """many blocks with a wide FFN: the FFN down-projections alone are split, into more merge blocks
    than there are counters; that refresh runs unsplit, and lora's split"""
    blocks, splits = refresh(host, block(64, 2048) * 120, 1)
    assert set(splits) == {1}
    blocks, splits = refresh(host, block(64, 2048) * 120, 0)
    assert blocks == 9480 and max(splits) == 3
    r = random.Random(9)
    for _ in range(500):
        dim = 64 * r.randint(1, 8)
        shapes = block(dim, 64 * r.randint(1, 64)) * r.randint(1, 200)
        blocks, splits = refresh(host, shapes, 1)
        assert blocks <= COUNTERS or max(splits) == 1
        for (i, _), s in zip(shapes, splits):   # every split has columns
            nc = i // 64
            assert (s - 1) * -(-nc // s) < nc
