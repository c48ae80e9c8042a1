"""The rules by which a call picks its kernels and sizes its memory (host code)."""
import ctypes
import os
import re
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "tests", "hostcheck", "route.cpp")
HDR = os.path.join(ROOT, "fastqsl_amd", "csrc", "fqsl_route.h")


@pytest.fixture(scope="module")
def route(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("route") / "libroute.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-fPIC", "-shared", "-I" + os.path.dirname(HDR),
                    SRC, "-o", so], check=True)
    return ctypes.CDLL(so)


@pytest.mark.parametrize("lines", [0, 1, 65536, 65537, 2 ** 24, 2 ** 24 + 1, 33554432, 2 ** 32 - 1, 2 ** 32])
def test_every_line_a_plain_trace_may_mark_has_its_place(route, lines):
    f = route.rt_plain_listed_lines
    f.restype = ctypes.c_ulonglong
    f.argtypes = [ctypes.c_int, ctypes.c_ulonglong, ctypes.c_int]
    # a count that only the device knows: no list, since `lines` bounds nothing
    assert f(1, lines, 0) == 0 and f(0, lines, 0) == 0
    # RK4 lines have no tangent class
    assert f(0, lines, 1) == 0
    # a counted RKF45 launch lists all its lines or none; line numbers are 32 bits wide
    assert f(1, lines, 1) == (lines if 65536 < lines < 2 ** 32 else 0)


@pytest.mark.parametrize("quad_lines", [0, 5, 20, 60, 10 ** 9])
@pytest.mark.parametrize("seed", range(20))
def test_launches_of_a_batch_share_no_counter(route, quad_lines, seed):
    """Layouts launched whole and layouts launched by field and method in one
    batch: every launch has its own work counter, inside the workspace's, and
    every request lies in one launch."""
    rng = np.random.default_rng(seed)
    m = int(rng.integers(1, 12))
    kind = np.sort(rng.integers(0, 3, m)).astype(np.int32)
    other = rng.integers(0, 2, m).astype(np.int8)
    other[0] = 1
    n = rng.integers(0, 20, m).astype(np.uint64)
    args = [m, kind.ctypes.data_as(ctypes.c_void_p), other.ctypes.data_as(ctypes.c_void_p), n.ctypes.data_as(ctypes.c_void_p)]
    counter, first = np.empty(m, np.int32), np.empty(m, np.int32)
    lines = np.empty(m, np.uint64)
    k = route.rt_batch_launches(*args, ctypes.c_ulonglong(quad_lines), counter.ctypes.data_as(ctypes.c_void_p),
                                first.ctypes.data_as(ctypes.c_void_p), lines.ctypes.data_as(ctypes.c_void_p))
    counter, first, lines = counter[:k], first[:k], lines[:k]
    assert len(set(counter)) == k and counter.min() >= 0 and counter.max() < route.rt_batch_groups(*args)
    assert list(first) == sorted(first) and first[0] == 0
    edges = list(first) + [m]
    assert [n[a:b].sum() for a, b in zip(edges[:-1], edges[1:])] == list(lines)


@pytest.mark.parametrize("out,expected", [([], 0), ([0, 0], 0), ([40, 0, 50], 0), ([10], 1), ([0, 40, 30], 1),
                                          ([40, 20, 50], 1), ([11, 14], 0)])
def test_results_over_the_seeds_are_seen(route, out, expected):
    """Addresses of the result arrays against seeds at 10, 20 and 30; 0 is NULL."""
    seeds = (ctypes.c_void_p * 3)(10, 20, 30)
    arr = (ctypes.c_void_p * max(1, len(out)))(*out)
    assert route.rt_plain_in_place(seeds, 3, arr, len(out)) == expected


def test_captured_per_line_launches_hold_no_work_counter(route):
    for in_place in (0, 1):
        for per_line in (0, 1):
            for capturing in (0, 1):
                got = route.rt_plain_by_lines(in_place, per_line, capturing)
                assert got == (1 if in_place or (per_line and capturing) else 0)


@pytest.mark.parametrize("code,ok_at,has_blocks,expected,calls", [
    (2, 1, 1, 0, 1),    # there is room
    (2, 2, 1, 0, 2),    # room once the kept blocks are given back
    (2, 3, 1, 2, 2),    # not even then
    (2, 2, 0, 2, 1),    # nothing to give back
    (7, 2, 1, 7, 1),    # another error
])
def test_allocations_find_kept_memory(route, code, ok_at, has_blocks, expected, calls):
    n = ctypes.c_int()
    assert route.rt_alloc_or_give_back(2, code, ok_at, has_blocks, ctypes.byref(n)) == expected
    assert n.value == calls


def test_every_device_allocation_may_find_kept_memory():
    src = open(os.path.join(ROOT, "fastqsl_amd", "csrc", "fqsl_kernels.hip")).read()
    src = re.sub(r"//[^\n]*|\"[^\"\n]*\"", "", src)
    bare = re.findall(r"[^\n]*\bhipMalloc(?:Async|Managed|FromPoolAsync)?\([^\n]*", src)
    inside = [l for l in bare if "return hipMalloc" in l and "[&] {" in l]
    assert len(inside) == 3 and bare == inside, bare


def test_fp64_work_that_goes_by_quads(route):
    f = route.rt_scott_fp64_quad_work
    f.restype, f.argtypes = ctypes.c_ulonglong, [ctypes.c_ulonglong]
    assert f(24 * 64 ** 3) == f(32 << 20) == 19000
    assert f((32 << 20) + 1) == f(24 * 256 ** 3) == 34000


def test_batches_by_quads(route):
    u = ctypes.c_ulonglong
    for rkf45, rk4, quads in ((0, 0, 1), (2 ** 23, 0, 1), (2 ** 23 + 1, 0, 0), (0, 2 ** 24, 1), (0, 2 ** 24 + 2, 0),
                              (2 ** 22, 2 ** 23, 1), (2 ** 22 + 1, 2 ** 23, 0)):
        assert route.rt_batch_fp32_by_quads(u(rkf45), u(rk4)) == quads, (rkf45, rk4)
    for lines, groups, rk4, quads in ((20000, 1, 1, 1), (20001, 1, 1, 0), (32768, 1, 0, 1), (32769, 1, 0, 0),
                                      (65536, 2, 1, 1), (65537, 2, 0, 0), (65536, 12, 0, 1)):
        assert route.rt_batch_fp64_by_quads(u(lines), groups, rk4) == quads, (lines, groups, rk4)
