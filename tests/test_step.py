"""The side tracers' step controller against its written expressions (CPU build)."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
N = 1 << 20


@pytest.fixture(scope="module")
def step(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("step") / "libstep.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-ffp-contract=off", "-fPIC", "-shared",
                    "-I" + os.path.join(ROOT, "fastqsl_amd", "csrc"),
                    os.path.join(ROOT, "tests", "hostcheck", "step.cpp"), "-o", so], check=True)
    return ctypes.CDLL(so)


def _p(a):
    return a.ctypes.data_as(ctypes.c_void_p)


# tolerances and squared error norms of traces, and the whole range of the fast path
@pytest.mark.parametrize("lo_tol,hi_tol,lo_e,hi_e", [(-12, -1, -22, 2), (-59.9, 5.9, -59.9, 59.9)])
@pytest.mark.parametrize("bits", [22, 23, 26, 52])
def test_argument_is_rounded_as_written(step, lo_tol, hi_tol, lo_e, hi_e, bits):
    rng = np.random.default_rng(bits + int(hi_e))
    tol = 10.0 ** rng.uniform(lo_tol, hi_tol, N)
    e2 = 10.0 ** rng.uniform(lo_e, hi_e, N)
    e2[: N // 4] = np.ldexp(rng.integers(1 << 52, 1 << 53, N // 4).astype(float), rng.integers(-150, 60, N // 4))
    e2[N // 4: N // 4 + 1000] = 4.0 ** rng.integers(-60, 60, 1000) * rng.integers(1, 100, 1000) ** 2.0   # exact roots
    eps = rng.uniform(-1, 1, N) * 2.0 ** -bits
    eps[::3] = np.where(rng.random(len(eps[::3])) < 0.5, 1, -1) * 2.0 ** -bits
    got, written, plain = np.empty(N), np.empty(N), np.empty(N, np.int32)
    step.st_arguments(ctypes.c_long(N), _p(tol), _p(e2), _p(eps), _p(got), _p(written), _p(plain))
    assert plain.all() and got.max() < 1e35      # in range of float
    np.testing.assert_array_equal(got, written)


def test_extreme_values_go_as_written(step):
    v = np.array([0.0, 1e-310, 1e-300, 1e-61, 1e61, 1e300, np.inf, np.nan, -1.0])
    other = np.full(v.size, 1e-3)
    plain, d = np.ones(v.size, np.int32), np.empty(v.size)
    for tol, e2 in ((other, v), (v, other), (v, v)):
        step.st_arguments(ctypes.c_long(v.size), _p(tol.copy()), _p(e2.copy()), _p(np.zeros(v.size)), _p(d.copy()),
                          _p(d), _p(plain))
        assert not plain.any()


# steps of a trace lie in [0.1, 100]; the first one is the caller's, and of the reference-
# shaped calls any float
@pytest.mark.parametrize("lo_s,hi_s", [(-1, 2), (-30, 38)])
@pytest.mark.parametrize("lo_q,hi_q", [(-6, 6), (-20, 34)])
def test_steps_are_those_of_the_exact_root(step, lo_s, hi_s, lo_q, hi_q):
    rng = np.random.default_rng(hi_s + hi_q)
    q = 10.0 ** rng.uniform(lo_q, hi_q, N)
    q[: N // 4] = (0.618 * (1 + rng.uniform(-3e-3, 3e-3, N // 4))) ** 5        # about the rejection
    s = 10.0 ** rng.uniform(lo_s, hi_s, N)
    s[N // 8: N // 4] = 100.0 / q[N // 8: N // 4] ** 0.2 * (1 + rng.uniform(-2e-3, 2e-3, N // 4 - N // 8))   # about both bounds
    s[N // 4: N // 2] = 0.1 / q[N // 4: N // 2] ** 0.2 * (1 + rng.uniform(-2e-3, 2e-3, N // 2 - N // 4))
    s[5], s[6] = 0.0, np.nan
    tol = 10.0 ** rng.uniform(-8, 5, N)
    e2 = (tol / q / 11.09) ** 2
    e2[7], e2[8], e2[9] = 0.0, np.nan, np.inf
    eps, eps5 = rng.uniform(-1, 1, N) * 2.0 ** -22, rng.uniform(-1, 1, N) * 1e-5
    got, written = np.empty(N), np.empty(N)
    ok, wok = np.empty(N, np.int32), np.empty(N, np.int32)
    step.st_steps(ctypes.c_long(N), _p(s), _p(tol), _p(e2), _p(eps), _p(eps5), _p(got), _p(ok), _p(written), _p(wok))
    np.testing.assert_array_equal(ok, wok)
    np.testing.assert_array_equal(got, written)
