"""Scott lines traced by quads of lanes give the bits of one lane a line.

The persistent schedule traces FP32c lines, and FP64 launches of a moderate
size, with one axis a lane; the per-line schedule runs one thread a line.  Both
must agree bit for bit in every output, whatever the launch's size (remainders
of a quad, a wavefront and a workgroup; refills; the ordered and the unordered
queue), with seeds on faces, below and outside the box and at NaN among them.
"""
import numpy as np
import pytest

from fastqsl_amd import synth

pytestmark = pytest.mark.gpu

LINES = 70000   # more than the quads of one full launch
CUTS = (0, 1, 2, 3, 5, 8, 15, 16, 17, 33, 64, 65, 255, 1023, 4097, 20000)


@pytest.fixture(scope="module")
def torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _seeds(shape):
    rng = np.random.default_rng(6)
    hi = np.array(shape, float) - 1
    p = hi * rng.uniform(-0.02, 1.02, (LINES, 3))
    p[: LINES // 2, 2] = 0.0                      # the usual seed plane
    p[LINES // 2: LINES // 2 + 500] = np.round(p[LINES // 2: LINES // 2 + 500])   # on grid planes
    p[7] = np.nan
    p[11, 1] = np.nan
    p[12], p[13] = 0.0, hi
    p[14, 0] = hi[0]
    p[15] = hi + 50.0
    p[16, 2] = -0.5
    p[17] = (1e9, -1e9, 3.0)
    return p.astype(np.float32)


@pytest.mark.parametrize("method", ["rkf45", "rk4"])
@pytest.mark.parametrize("layout,precision,twist", [("cell32", "fp32c", False), ("soa32", "fp32c", False),
                                                    ("soa64", "fp64", False), ("cell32", "fp32c", True),
                                                    ("soa32", "fp32c", True), ("soa64", "fp64", True)])
def test_quads_equal_one_thread_per_line(torch, layout, precision, twist, method):
    import fastqsl_amd as fq
    from fastqsl_amd import postproc
    shape = (26, 21, 17)
    b = synth.multipole(shape, seed=3, count=12, device="cpu")
    current = postproc.curl_index(*b) if twist else None
    p = _seeds(shape)
    x, y, z = (torch.as_tensor(np.ascontiguousarray(p[:, i])).cuda() for i in range(3))
    names = fq.trace.SCOTT_OUTPUTS + (("twist",) if twist else ())
    kw = dict(method=method, step=0.25, tol=1e-5, precision=precision, outputs=names)
    with fq.Field(*b, layouts=(layout,), current=current) as f:
        ref = fq.trace_scott(f, x, y, z, schedule="per_line", **kw)
        ref = {k: ref[k].cpu().numpy() for k in names}
        assert int((ref["flag_end"] > 0).sum()) > LINES // 2
        edges = [0, LINES] + list(np.cumsum(CUTS))
        for a, e in zip(edges[:-1], edges[1:]):
            if a >= e:
                continue
            part = fq.trace_scott(f, x[a:e], y[a:e], z[a:e], schedule="persistent", **kw)
            torch.cuda.synchronize()
            for k in names:
                np.testing.assert_array_equal(part[k].cpu().numpy(), ref[k][a:e], err_msg=f"{k} of lines {a}..{e}")
