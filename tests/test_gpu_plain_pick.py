"""Large RK4 plain traces on component arrays, of which the seeds pick the kernel.

Lines close together (one side a lane) and lines anywhere in the box (quads, one
wavefront a SIMD), at the counts where each begins: the bits of the 4-byte
results are those of calls of a few thousand lines.
"""
import numpy as np
import pytest

from fastqsl_amd import synth

pytestmark = pytest.mark.gpu

SHAPE = (26, 21, 17)


@pytest.mark.parametrize("kind", ["volume", "map"])
@pytest.mark.parametrize("n", [16383, 16384, 65535, 65536, 200001])
@pytest.mark.parametrize("layout,precision", [("soa64", "fp64"), ("soa32", "fp32c")])
def test_large_calls_equal_small_ones(layout, precision, n, kind):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import fastqsl_amd as fq
    b = synth.multipole(SHAPE, seed=3, count=12, device="cpu")
    hi = np.array(SHAPE, float) - 1
    if kind == "volume":
        p = np.random.default_rng(1).uniform(-0.02, 1.02, (n, 3)) * hi
    else:
        t = np.arange(n)
        p = np.column_stack([(t % 400) / 400 * hi[0], (t // 400) / (n // 400 + 1) * hi[1], np.full(n, 1e-3)])
    p[7], p[9, 1], p[11] = np.nan, np.nan, hi + 50.0
    x, y, z = (torch.as_tensor(np.ascontiguousarray(p[:, i], dtype=np.float32)).cuda() for i in range(3))
    names = tuple(k for k in fq.trace.PLAIN_OUTPUTS if k != "line_len")
    kw = dict(method="rk4", step=0.25, precision=precision, outputs=names)
    with fq.Field(*b, layouts=(layout,)) as f:
        whole = fq.trace_plain(f, x, y, z, **kw)
        only = fq.trace_plain(f, x, y, z, **dict(kw, outputs=("end_x", "end_y", "end_z")))
        torch.cuda.synchronize()
        for k in ("end_x", "end_y", "end_z"):
            np.testing.assert_array_equal(only[k].cpu().numpy(), whole[k].cpu().numpy(), err_msg=k)
        for a in (0, n // 2, n - 3000):
            part = fq.trace_plain(f, *[v[a:a + 3000].clone() for v in (x, y, z)], **kw)
            torch.cuda.synchronize()
            for k in names:
                np.testing.assert_array_equal(part[k].cpu().numpy(), whole[k][a:a + 3000].cpu().numpy(), err_msg=k)
