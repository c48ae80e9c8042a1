"""The plain tracer's two ways to lay lines over lanes give the same bits.

A launch of few sides is traced by quads of lanes (one axis a lane); a large
RKF45 launch traces the lines nearly tangent to the plane by quads and all
others one side per lane.  The same seeds in one large call and in calls of 1
to a few thousand lines (remainders of a quad, a wavefront and a workgroup)
must agree bit for bit, for every field layout and geometry, with seeds
outside the box, on its faces and at NaN among them.
"""
import numpy as np
import pytest

from fastqsl_amd import synth

pytestmark = pytest.mark.gpu

LINES = 66000   # > 65,536 lines: two sides each pass the quads' limit
CUTS = (0, 1, 2, 3, 5, 8, 15, 16, 17, 33, 64, 65, 128, 255, 511, 1023, 4097, 9000)


@pytest.fixture(scope="module")
def torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _seeds(shape, axes, seed):
    rng = np.random.default_rng(seed)
    lo = np.array([0.0, 0.0, 0.0]) if axes is None else np.array([a[0] for a in axes], float)
    hi = np.array(shape, float) - 1 if axes is None else np.array([a[-1] for a in axes], float)
    p = lo + (hi - lo) * rng.uniform(-0.02, 1.02, (LINES, 3))
    p[: LINES // 2, 2] = lo[2] + 1e-4 * (hi[2] - lo[2])          # the usual seed plane
    p[7] = np.nan
    p[11, 1] = np.nan
    p[12], p[13] = lo, hi
    p[14, 0] = hi[0]
    p[15] = hi + 50.0
    return p.astype(np.float32)


@pytest.mark.parametrize("layout,precision", [("cell32", "fp32c"), ("soa32", "fp32c"), ("soa64", "fp64")])
@pytest.mark.parametrize("method,stretched", [("rkf45", False), ("rk4", False), ("rkf45", True)])
def test_large_launch_equals_small_ones(torch, layout, precision, method, stretched):
    import fastqsl_amd as fq
    shape = (26, 21, 17)
    axes = None
    if stretched:
        b, axes = synth.stretched_multipole(shape, seed=3, count=12, scale=10.0, device="cpu")
    else:
        b = synth.multipole(shape, seed=3, count=12, device="cpu")
    p = _seeds(shape, axes, 4)
    x, y, z = (torch.as_tensor(np.ascontiguousarray(p[:, i])).cuda() for i in range(3))
    kw = dict(method=method, step=0.25 if axes is None else 0.05, tol_coef=0.3, precision=precision)
    with fq.Field(*b, layouts=(layout,), axes=axes) as f:
        whole = fq.trace_plain(f, x, y, z, **kw)
        torch.cuda.synchronize()
        assert int((whole["flag_end"] > 0).sum()) > LINES // 2
        edges = list(np.cumsum(CUTS)) + [LINES]
        for a, e in zip(edges[:-1], edges[1:]):
            if a == e:
                continue
            part = fq.trace_plain(f, x[a:e], y[a:e], z[a:e], **kw)
            torch.cuda.synchronize()
            for k in fq.trace.PLAIN_OUTPUTS:
                u, v = part[k].cpu().numpy(), whole[k][a:e].cpu().numpy()
                np.testing.assert_array_equal(u, v, err_msg=f"{k} of lines {a}..{e}")
