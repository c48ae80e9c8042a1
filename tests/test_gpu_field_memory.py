"""Fields built in memory that an earlier field gave back hold the same data.

A destroyed field's large blocks serve the next fields whose layouts fit them;
a trace on such a field must give the bits of the same field built first, with
a larger and a smaller field before it, while another field is alive, and from
float and double input.
"""
import numpy as np
import pytest

from fastqsl_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("shape", [(65, 64, 50), (97, 63, 41), (258, 33, 17), (2, 300, 130)])
def test_rebuilt_field_traces_the_same_bits(shape, dtype):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import fastqsl_amd as fq
    b = [c.astype(dtype) for c in synth.multipole(shape, seed=2, count=10, device="cpu")]
    rng = np.random.default_rng(0)
    p = (rng.uniform(0.02, 0.98, (3000, 3)) * (np.array(shape) - 1)).astype(np.float32)

    def trace(f):
        r = fq.trace_scott(f, p[:, 0], p[:, 1], p[:, 2], tol=1e-5)
        torch.cuda.synchronize()
        return {k: v.cpu().numpy() for k, v in r.items() if k != "_seeds"}

    with fq.Field(*b) as f:
        first = trace(f)
    for grow in (0, 2, -1):
        other = tuple(max(2, n + grow) for n in shape)
        fq.Field(*synth.multipole(other, seed=9, count=4, device="cpu")).close()
        with fq.Field(*synth.multipole(shape, seed=8, count=4, device="cpu")) as alive, fq.Field(*b) as f:
            again = trace(f)
            assert not np.array_equal(trace(alive)["line_len"], first["line_len"])
        for k, v in first.items():
            np.testing.assert_array_equal(again[k], v, err_msg=k)
