"""The rules by which a call picks its kernels and sizes its memory (host code)."""
import ctypes
import os
import subprocess

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
