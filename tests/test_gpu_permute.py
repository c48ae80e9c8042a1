"""Per-line arrays into an order and back, all in one launch, against torch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,count", [(0, 3), (1, 1), (63, 24), (256, 5), (257, 25), (70001, 49)])
def test_permute_equals_torch_indexing(n, count):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from fastqsl_amd.qmap import _permute
    rng = np.random.default_rng(n + count)
    perm = torch.as_tensor(rng.permutation(n).astype(np.int32)).cuda()
    kinds = (torch.float32, torch.int32, torch.float64)
    arrays = []
    for k in range(count):
        v = torch.as_tensor(rng.integers(-1000, 1000, (n, 3)) / 8.0).to(kinds[k % 3]).cuda()
        arrays.append(v[:, k % 3] if k % 2 else v[:, 0].contiguous())
    idx = perm.long()
    for v, g in zip(arrays, _permute(arrays, perm, scatter=False)):
        assert g.is_contiguous() and torch.equal(g, v[idx])
    for v, g in zip(arrays, _permute(arrays, perm, scatter=True)):
        u = torch.empty_like(v)
        u[idx] = v
        assert g.is_contiguous() and torch.equal(g, u)


def test_more_arrays_than_a_launch_takes_are_refused():
    from fastqsl_amd import _lib
    with pytest.raises(_lib.FqslError, match="at most 24"):
        _lib.check(_lib.lib().fqsl_permute(1, None, 0, 25, None, None, None, None, None))
