"""The reference-shaped plain entries at every line count.

The count lives on the device: the entries read it where they wait for the
twist switch anyway, and leave it there where the switch is NULL.  Both must
give the bits of the handle entry on the same in-place field, below and above
the count from which tangent lines are listed; a call of more than 2^24 lines
must give its last lines as a call of those alone does.
"""
import ctypes

import numpy as np
import pytest

from fastqsl_amd import synth

pytestmark = pytest.mark.gpu

SHAPE = (26, 21, 17)
OUT = ("start_x", "start_y", "start_z", "flag_start", "end_x", "end_y", "end_z", "flag_end", "b_this_x", "b_this_y",
       "b_this_z", "b_flag", "b_start_x", "b_start_y", "b_start_z", "b_end_x", "b_end_y", "b_end_z")


@pytest.fixture(scope="module")
def torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _call(torch, b, axes, x, y, z, method, with_flag, n=None):
    """One call of the C entry; with_flag: pass the twist switch (off) or NULL."""
    from fastqsl_amd import _lib
    n = x.numel() if n is None else n
    t = lambda a, dt: torch.as_tensor(np.ascontiguousarray(a), dtype=dt, device="cuda")  # noqa: E731
    keep = [t(np.asarray(c, np.float32).ravel(order="F"), torch.float32) for c in b]
    keep.append(t(b[0].shape, torch.int32))
    if axes is not None:
        keep += [t(a, torch.float32) for a in axes] + [torch.tensor([False], device="cuda")]
    out = {k: torch.full((x.numel(),), -7, dtype=torch.int32 if "flag" in k else torch.float32, device="cuda") for k in OUT}
    flag = torch.tensor([False], device="cuda")
    rest = [t([0.0, 0.0, 1.0], torch.float32)]
    tail = [t([0.25 if axes is None else 0.05], torch.float32), t([n], torch.int64),
            torch.full((x.numel(),), -7, dtype=torch.float64, device="cuda"), t([0.3], torch.float32)]
    ptr = lambda a: ctypes.c_void_p(a.data_ptr())  # noqa: E731
    args = [ptr(a) for a in keep] + [None] * 4 + [ptr(flag) if with_flag else None]
    args += [ptr(a) for a in (x, y, z)] + [ptr(a) for a in rest] + [ptr(out[k]) for k in OUT] + [ptr(a) for a in tail]
    args += [0, 0, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)]
    L = _lib.lib()
    if axes is not None:
        rc = L.fqsl_TraceAllBlineStretch(*args)
    else:
        rc = L.fqsl_TraceAllBline(_lib.METHODS[method], *args)
    _lib.check(rc)
    torch.cuda.synchronize()
    return dict({k: out[k].cpu().numpy() for k in OUT}, line_len=tail[2].cpu().numpy())


def _problem(torch, stretched, n):
    rng = np.random.default_rng(4)
    if stretched:
        b, axes = synth.stretched_multipole(SHAPE, seed=3, count=12, scale=10.0, device="cpu")
        axes = [np.asarray(a, np.float32) for a in axes]
        lo, hi = np.array([a[0] for a in axes], float), np.array([a[-1] for a in axes], float)
    else:
        b, axes = synth.multipole(SHAPE, seed=3, count=12, device="cpu"), None
        lo, hi = np.zeros(3), np.array(SHAPE, float) - 1
    p = lo + (hi - lo) * rng.uniform(0.0, 1.0, (n, 3))
    p[: n // 2, 2] = lo[2] + 1e-4 * (hi[2] - lo[2])
    return b, axes, [torch.as_tensor(np.ascontiguousarray(p[:, i], dtype=np.float32)).cuda() for i in range(3)]


@pytest.mark.parametrize("with_flag", [True, False])
@pytest.mark.parametrize("n", [0, 1, 65536, 65537, 70001])
@pytest.mark.parametrize("method,stretched", [("rkf45", False), ("rk4", False), ("rkf45", True)])
def test_counts_give_the_bits_of_the_handle_entry(torch, method, stretched, n, with_flag):
    import fastqsl_amd as fq
    b, axes, (x, y, z) = _problem(torch, stretched, max(n, 8))
    got = _call(torch, b, axes, x, y, z, method, with_flag, n=n)
    for k, v in got.items():
        assert (v[n:] == -7).all(), k      # nothing past the count is written
    if n == 0:
        return
    step = float(np.float32(0.25 if axes is None else 0.05))
    with fq.Field(*b, layouts=("soa32",), axes=axes, lookup="bisect") as f:
        ref = fq.trace_plain(f, x, y, z, method=method, step=step, tol_coef=float(np.float32(0.3)), precision="fp32c")
        torch.cuda.synchronize()
        for k, v in got.items():
            np.testing.assert_array_equal(v[:n], ref[k].cpu().numpy()[:n], err_msg=k)


@pytest.mark.parametrize("with_flag", [True, False])
def test_more_lines_than_two_to_the_24(torch, with_flag):
    n, m = 2 ** 24 + 70001, 4096
    b, _, part = _problem(torch, False, 1 << 16)
    xyz = [torch.cat([a.repeat(n // a.numel()), a[: n % a.numel()]]) for a in part]
    got = _call(torch, b, None, *xyz, "rkf45", with_flag)
    ref = _call(torch, b, None, *[a[n - m:].clone() for a in xyz], "rkf45", with_flag)
    for k, v in got.items():
        np.testing.assert_array_equal(v[n - m:], ref[k], err_msg=k)
