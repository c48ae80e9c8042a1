"""What is kept of closed fields' memory can be given back."""
import numpy as np
import pytest

from fastqsl_amd import synth

pytestmark = pytest.mark.gpu


def test_release_gives_the_memory_back_and_fields_still_work():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import fastqsl_amd as fq
    shape = (128, 128, 64)
    b = synth.multipole(shape, seed=2, count=6, device="cpu")
    p = (np.random.default_rng(0).uniform(0.02, 0.98, (500, 3)) * (np.array(shape) - 1)).astype(np.float32)

    def trace(f):
        r = fq.trace_scott(f, p[:, 0], p[:, 1], p[:, 2], tol=1e-4)
        torch.cuda.synchronize()
        return r["q_0"].cpu().numpy()

    fq.release_field_memory()
    with fq.Field(*b) as f:
        first, size = trace(f), f.nbytes
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    assert fq.release_field_memory(keep=1 << 40) >= size       # kept, and stays so
    assert torch.cuda.mem_get_info()[0] == free
    part = fq.release_field_memory(keep=size // 2)
    assert 0 < part <= size // 2
    assert fq.release_field_memory() == 0
    assert torch.cuda.mem_get_info()[0] >= free + size // 2
    with fq.Field(*b) as f:
        np.testing.assert_array_equal(trace(f), first)
