"""A batch that one launch traces gives the bits of one thread per line.

Requests of every method over fields of several shapes, some with cell records
and some without, so that quads of one wavefront trace lines of different fields,
steps and integrators; sizes at the edges of a quad, a wavefront and a workgroup,
empty requests, and more lines than one full launch holds.  FP64 batches on both
sides of the limit up to which quads trace them, and the mixed variant, which
keeps a launch per field and method.
"""
import numpy as np
import pytest

from fastqsl_amd import synth
from fastqsl_amd.trace import SCOTT_OUTPUTS

pytestmark = pytest.mark.gpu

SHAPES = ((20, 17, 15), (33, 12, 24), (9, 40, 11))
SIZES = (1, 2, 3, 4, 15, 16, 17, 0, 63, 65, 255, 257, 1025)


@pytest.fixture(scope="module")
def torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _request(torch, field, shape, k, n):
    rng = np.random.default_rng(100 + k)
    p = rng.uniform(-0.02, 1.02, (n, 3)) * (np.array(shape, float) - 1)
    p[: n // 2, 2] = 0.0
    if n > 16:
        p[5] = np.nan
        p[6, 2] = -0.5
    x, y, z = (torch.as_tensor(np.ascontiguousarray(p[:, i]).astype(np.float32)).cuda() for i in range(3))
    return dict(field=field, x=x, y=y, z=z, method=("rkf45", "rk4")[(k // 2) % 2], tol=(1e-5, 3e-6, 1e-6)[k % 3],
                step=(0.25, 0.5)[k % 2])


@pytest.mark.parametrize("precision,sizes", [("fp32c", SIZES), ("fp32c", SIZES + (70000, 40000)), ("fp32c", (3,)),
                                             ("fp32c", (0, 0)), ("mixed", SIZES), ("fp64", SIZES),
                                             ("fp64", SIZES + (90000, 60000))])
def test_batch_equals_one_thread_per_line(torch, precision, sizes):
    import fastqsl_amd as fq
    from fastqsl_amd.batch import ScottBatch
    layouts = [("soa64", "cell32"), ("soa64", "soa32"), ("soa64", "cell32")]
    fields = [fq.Field(*synth.multipole(s, seed=3 + i, count=10, device="cpu"), layouts=layouts[i])
              for i, s in enumerate(SHAPES)]
    try:
        reqs = [_request(torch, fields[k % 3], SHAPES[k % 3], k, n) for k, n in enumerate(sizes)]
        with ScottBatch(reqs, precision=precision, outputs=SCOTT_OUTPUTS) as b:
            for _ in range(2):
                b.run()
            torch.cuda.synchronize()
            times = b.times_ms()
            for k, (rq, res) in enumerate(zip(reqs, b.results)):
                assert (times[k] > 0) == (sizes[k] > 0)
                if sizes[k] == 0:
                    continue
                ref = fq.trace_scott(rq["field"], rq["x"], rq["y"], rq["z"], method=rq["method"], step=rq["step"],
                                     tol=rq["tol"], precision=precision, schedule="per_line")
                for name in SCOTT_OUTPUTS:
                    np.testing.assert_array_equal(res[name].cpu().numpy(), ref[name].cpu().numpy(),
                                                  err_msg=f"{name} of request {k}")
    finally:
        for f in fields:
            f.close()
