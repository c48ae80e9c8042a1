"""Plain traces whose results lie on the seed arrays.

One thread traces both sides of such a line, with the one-lane code that the CPU
tests build.  The results kept in 4 bytes, and the length of FP32 lines, must
have the bits of the same call with separate arrays, which quads of lanes and
side tasks trace: below and above the count from which tangent lines are listed,
for every layout and geometry, with seeds outside the box, on its faces and at
NaN among them.  (The twist of the two sides is summed apart by the side tasks,
and FP64 lengths are fused with other products there.)  Whichever results lie on
the seeds, one thread a line gives the same bits of everything.
"""
import numpy as np
import pytest

from fastqsl_amd import synth

pytestmark = pytest.mark.gpu

SHAPE = (26, 21, 17)


@pytest.fixture(scope="module")
def torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _seeds(axes, n):
    rng = np.random.default_rng(7)
    lo = np.zeros(3) if axes is None else np.array([a[0] for a in axes], float)
    hi = np.array(SHAPE, float) - 1 if axes is None else np.array([a[-1] for a in axes], float)
    p = lo + (hi - lo) * rng.uniform(-0.02, 1.02, (n, 3))
    p[: n // 2, 2] = lo[2] + 1e-4 * (hi[2] - lo[2])
    if n > 8:
        p[1], p[2, 1], p[3], p[4], p[5], p[6, 0] = np.nan, np.nan, lo, hi, hi + 50.0, hi[0]
    return p.astype(np.float32)


@pytest.mark.parametrize("n,twist", [(65, True), (70001, False)])
@pytest.mark.parametrize("layout,precision", [("cell32", "fp32c"), ("soa32", "fp32c"), ("soa64", "fp64")])
@pytest.mark.parametrize("method,stretched", [("rkf45", False), ("rk4", False), ("rkf45", True)])
def test_results_over_the_seeds_equal_separate_arrays(torch, method, stretched, layout, precision, n, twist):
    import fastqsl_amd as fq
    axes = None
    if stretched:
        b, axes = synth.stretched_multipole(SHAPE, seed=3, count=12, scale=10.0, device="cpu")
    else:
        b = synth.multipole(SHAPE, seed=3, count=12, device="cpu")
    cur = (b[1], b[2], b[0]) if twist else None      # any field serves as the current
    p = _seeds(axes, n)
    names = fq.trace.PLAIN_OUTPUTS + ("evals",) + (("twist",) if twist else ())
    names = tuple(dict.fromkeys(names))
    kw = dict(method=method, step=0.25 if axes is None else 0.05, tol_coef=3.0, precision=precision, outputs=names)
    fresh = lambda: [torch.as_tensor(np.ascontiguousarray(p[:, i])).cuda() for i in range(3)]  # noqa: E731
    with fq.Field(*b, layouts=(layout,), axes=axes, current=cur) as f:
        ref = fq.trace_plain(f, *fresh(), **kw)
        torch.cuda.synchronize()
        sides = [k for k in names if k != "twist" and not (k == "line_len" and precision == "fp64")]
        ref, first = {k: ref[k].cpu().numpy() for k in sides}, None
        for over in (("start_x", "start_y", "start_z"), ("b_this_x", "flag_end", None)):
            xyz = fresh()
            out = {k: (a.view(torch.int32) if k.startswith("flag") else a)
                   for k, a in zip(over, xyz) if k}
            got = fq.trace_plain(f, *xyz, out=out, **kw)
            torch.cuda.synchronize()
            for k, a in zip(over, xyz):
                assert k is None or got[k].data_ptr() == a.data_ptr()
            got = {k: got[k].cpu().numpy() for k in names}
            first = first or got
            for k in names:
                np.testing.assert_array_equal(got[k], first[k], err_msg=f"{k}, results over the seeds: {over}")
            for k in sides:
                np.testing.assert_array_equal(got[k], ref[k], err_msg=f"{k}, results over the seeds: {over}")
