"""A batch whose layouts are traced in different ways traces every line.

More FP32c lines than a batch takes by quads, over fields with cell records and
in two (field, method) groups, beside requests on a field without cells, which
go by quads: each request must give the bits of its own trace.
"""
import numpy as np
import pytest

from fastqsl_amd import synth

pytestmark = pytest.mark.gpu

NAMES = ("q_0", "q_perp", "flag_start", "flag_end", "line_len", "evals")


def test_large_cell_layout_beside_a_small_one_without_cells():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import fastqsl_amd as fq
    from fastqsl_amd.batch import ScottBatch
    shape, big, small = (9, 8, 7), 2 ** 23 + 1025, 3001
    b = synth.multipole(shape, seed=3, count=8, device="cpu")
    rng = np.random.default_rng(5)

    def seeds(n):
        p = torch.as_tensor((rng.uniform(0.0, 1.0, (4096, 3)) * (np.array(shape) - 1)).astype(np.float32)).cuda()
        return [p[:, i].repeat(-(-n // 4096))[:n].contiguous() for i in range(3)]

    with fq.Field(*b, layouts=("cell32",)) as cells, fq.Field(*b, layouts=("soa32",)) as arrays:
        reqs = []
        for field, n, method in ((cells, big, "rk4"), (arrays, small, "rkf45"), (cells, big, "rkf45"),
                                 (arrays, small, "rk4")):
            x, y, z = seeds(n)
            reqs.append(dict(field=field, x=x, y=y, z=z, method=method, step=0.5, tol=1e-4))
        with ScottBatch(reqs, precision="fp32c", outputs=NAMES) as batch:
            for _ in range(2):
                for r in batch.results:
                    for v in r.values():
                        v.fill_(-7)
                batch.run()
            torch.cuda.synchronize()
            assert all(t > 0 for t in batch.times_ms())
            for k, (rq, res) in enumerate(zip(reqs, batch.results)):
                n = rq["x"].numel()
                for part in (slice(0, min(n, 5000)), slice(max(0, n - 5000), n)):
                    ref = fq.trace_scott(rq["field"], *[rq[a][part].clone() for a in "xyz"], method=rq["method"],
                                         step=0.5, tol=1e-4, precision="fp32c", schedule="per_line", outputs=NAMES)
                    for name in NAMES:
                        np.testing.assert_array_equal(res[name][part].cpu().numpy(), ref[name].cpu().numpy(),
                                                      err_msg=f"{name} of request {k}")
                    assert int((ref["flag_end"] > 0).sum()) > 0


@pytest.mark.parametrize("method,n", [("rk4", 20000), ("rk4", 20001), ("rkf45", 32768), ("rkf45", 32769)])
def test_one_fp64_request_on_both_sides_of_its_rule(method, n):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import fastqsl_amd as fq
    from fastqsl_amd.batch import ScottBatch
    shape = (20, 17, 15)
    rng = np.random.default_rng(2)
    p = torch.as_tensor((rng.uniform(-0.02, 1.02, (n, 3)) * (np.array(shape) - 1)).astype(np.float32)).cuda()
    x, y, z = (p[:, i].contiguous() for i in range(3))
    with fq.Field(*synth.multipole(shape, seed=3, count=8, device="cpu"), layouts=("soa64",)) as f:
        rq = dict(field=f, x=x, y=y, z=z, method=method, step=0.25, tol=1e-5)
        ref = fq.trace_scott(f, x, y, z, method=method, step=0.25, tol=1e-5, precision="fp64", schedule="per_line",
                             outputs=NAMES)
        with ScottBatch([rq], precision="fp64", outputs=NAMES) as batch:
            for _ in range(2):
                batch.run()
            torch.cuda.synchronize()
            for name in NAMES:
                np.testing.assert_array_equal(batch.results[0][name].cpu().numpy(), ref[name].cpu().numpy(), err_msg=name)
