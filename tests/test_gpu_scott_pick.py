"""FP64 RK4 launches of which the lines' estimated lengths pick the kernel.

Seeds anywhere in the box (many long lines: one line per lane) and seeds on a
plane with few long lines (by quads of lanes), at the counts where the choice
begins and ends: the bits are those of one thread per line.
"""
import numpy as np
import pytest

from fastqsl_amd import synth

pytestmark = pytest.mark.gpu

SHAPE = (24, 22, 18)


@pytest.mark.parametrize("kind", ["volume", "plane"])
@pytest.mark.parametrize("twist", [False, True])
@pytest.mark.parametrize("n", [19000, 19001, 40000, 65536, 65537])
def test_picked_kernel_gives_the_bits_of_one_thread_per_line(n, kind, twist):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import fastqsl_amd as fq
    b = synth.multipole(SHAPE, seed=3, count=12, device="cpu")
    rng = np.random.default_rng(n)
    p = rng.uniform(0.0, 1.0, (n, 3)) * (np.array(SHAPE) - 1)
    if kind == "plane":
        p[:, 2] = 0.0
        p[: n - 50, :2] = p[: n - 50, :2] * 0.05       # nearly all lines start in one corner
    p[3], p[5, 2] = np.nan, -0.5
    x, y, z = (torch.as_tensor(np.ascontiguousarray(p[:, i], dtype=np.float32)).cuda() for i in range(3))
    names = fq.trace.SCOTT_OUTPUTS + (("twist",) if twist else ())
    kw = dict(method="rk4", step=0.25, precision="fp64", outputs=names)
    with fq.Field(*b, layouts=("soa64",), current=(b[1], b[2], b[0]) if twist else None) as f:
        ref = fq.trace_scott(f, x, y, z, schedule="per_line", **kw)
        for _ in range(2):
            got = fq.trace_scott(f, x, y, z, schedule="persistent", **kw)
            torch.cuda.synchronize()
            for k in names:
                np.testing.assert_array_equal(got[k].cpu().numpy(), ref[k].cpu().numpy(), err_msg=k)


@pytest.mark.parametrize("kind", ["volume", "map"])
@pytest.mark.parametrize("n", [2 ** 20, 2 ** 20 + 1, 2 ** 20 + 300001])
def test_large_fp32c_rk4_launches(n, kind):
    """FP32c RK4 lines on cells: dense seeds by lanes, others by quads."""
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
        p = np.column_stack([(t % 1100) / 1100 * hi[0], (t // 1100) / (n // 1100 + 1) * hi[1], np.zeros(n)])
    p[7], p[9, 1], p[11], p[13, 2] = np.nan, np.nan, hi + 50.0, -0.5
    x, y, z = (torch.as_tensor(np.ascontiguousarray(p[:, i], dtype=np.float32)).cuda() for i in range(3))
    names = fq.trace.SCOTT_OUTPUTS
    kw = dict(method="rk4", step=0.5, precision="fp32c", outputs=names)
    with fq.Field(*b, layouts=("cell32",)) as f:
        got = fq.trace_scott(f, x, y, z, schedule="persistent", **kw)
        ref = fq.trace_scott(f, x, y, z, schedule="per_line", **kw)
        torch.cuda.synchronize()
        for k in names:
            assert torch.equal(got[k].view(torch.int32 if got[k].element_size() == 4 else torch.int64),
                               ref[k].view(torch.int32 if ref[k].element_size() == 4 else torch.int64)) or \
                np.array_equal(got[k].cpu().numpy(), ref[k].cpu().numpy(), equal_nan=True), k


@pytest.mark.parametrize("kind", ["volume", "map"])
@pytest.mark.parametrize("shape,n,method", [(SHAPE, 300000, "rkf45"), (SHAPE, 300001, "rkf45"), (SHAPE, 180000, "rk4"),
                                            (SHAPE, 180001, "rk4"),
                                            ((160, 140, 128), 65536, "rkf45"), ((160, 140, 128), 65537, "rkf45"),
                                            ((160, 140, 128), 300001, "rk4"), ((160, 140, 128), 1048577, "rk4")])
@pytest.mark.parametrize("twist", [False, True])
def test_component_arrays(shape, n, method, kind, twist):
    """FP32c lines on float component arrays: a field that the caches hold, or a larger one."""
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import fastqsl_amd as fq
    b = synth.multipole(shape, seed=3, count=12, device="cpu")
    hi = np.array(shape, float) - 1
    if kind == "volume":
        p = np.random.default_rng(1).uniform(-0.02, 1.02, (n, 3)) * hi
    else:
        t = np.arange(n)
        p = np.column_stack([(t % 1100) / 1100 * hi[0], (t // 1100) / (n // 1100 + 1) * hi[1], np.zeros(n)])
    p[7], p[9, 1], p[11], p[13, 2] = np.nan, np.nan, hi + 50.0, -0.5
    x, y, z = (torch.as_tensor(np.ascontiguousarray(p[:, i], dtype=np.float32)).cuda() for i in range(3))
    names = ("q_0", "q_perp", "start_x", "start_y", "start_z", "end_x", "end_y", "end_z", "flag_start", "flag_end", "evals")
    names += ("twist",) if twist else ()
    kw = dict(method=method, step=0.5, tol=1e-4, precision="fp32c", outputs=names)
    with fq.Field(*b, layouts=("soa32",), current=(b[1], b[2], b[0]) if twist else None) as f:
        ref = fq.trace_scott(f, x, y, z, schedule="per_line", **kw)
        for _ in range(2):
            got = fq.trace_scott(f, x, y, z, schedule="persistent", **kw)
            torch.cuda.synchronize()
            for k in names:
                assert np.array_equal(got[k].cpu().numpy(), ref[k].cpu().numpy(), equal_nan=True), k
