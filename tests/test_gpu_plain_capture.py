"""Captured plain traces give on every replay what the eager call gives.

The per-line schedule is captured as one thread per line, the persistent one by
quads of lanes; below and above the count from which an eager RKF45 call lists
its tangent lines.
"""
import numpy as np
import pytest

from fastqsl_amd import synth

pytestmark = pytest.mark.gpu

SHAPE = (26, 21, 17)


@pytest.mark.parametrize("schedule", ["per_line", "persistent"])
@pytest.mark.parametrize("method,stretched", [("rkf45", False), ("rk4", False), ("rkf45", True)])
@pytest.mark.parametrize("n", [257, 70001])
def test_replays_equal_the_eager_call(n, method, stretched, schedule):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import fastqsl_amd as fq
    axes = None
    if stretched:
        b, axes = synth.stretched_multipole(SHAPE, seed=3, count=12, scale=10.0, device="cpu")
    else:
        b = synth.multipole(SHAPE, seed=3, count=12, device="cpu")
    lo = np.zeros(3) if axes is None else np.array([a[0] for a in axes], float)
    hi = np.array(SHAPE, float) - 1 if axes is None else np.array([a[-1] for a in axes], float)
    rng = np.random.default_rng(9)
    sets = [torch.as_tensor((lo + (hi - lo) * rng.uniform(0.02, 0.98, (n, 3))).astype(np.float32)).cuda() for _ in range(3)]
    x, y, z = (sets[0][:, i].contiguous() for i in range(3))
    names = tuple(k for k in fq.trace.PLAIN_OUTPUTS)
    kw = dict(method=method, step=0.25 if axes is None else 0.05, tol_coef=3.0, schedule=schedule, outputs=names)
    with fq.Field(*b, axes=axes) as f:
        fq.trace_plain(f, x, y, z, **kw)     # first use outside the capture
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = fq.trace_plain(f, x, y, z, **kw)
        for s in sets:
            for a, i in ((x, 0), (y, 1), (z, 2)):
                a.copy_(s[:, i])
            for k in names:
                out[k].fill_(-7)
            graph.replay()
            torch.cuda.synchronize()
            got = {k: out[k].cpu().numpy() for k in names}
            ref = fq.trace_plain(f, x, y, z, **kw)
            torch.cuda.synchronize()
            for k in names:
                np.testing.assert_array_equal(got[k], ref[k].cpu().numpy(), err_msg=k)
