"""The reference-shaped Scott entry gives the bits of the in-place field.

Large fields with many lines are paired in x before they are traced; a line must
not depend on it.  Node counts around the smallest that is paired, lines on both
sides of the rule, seeds on faces, outside and at NaN, with the twist, called
twice and after a field of another size so that the pairs' memory is used again.
"""
import numpy as np
import pytest

from fastqsl_amd import synth

pytestmark = pytest.mark.gpu


def _call(torch, fq, b, cur, p, schedule):
    n = len(p)
    t = lambda a, dt: torch.as_tensor(np.ascontiguousarray(a), dtype=dt, device="cuda")  # noqa: E731
    flat = lambda c: t(np.asarray(c, np.float32).ravel(order="F"), torch.float32)  # noqa: E731
    f32 = lambda: torch.full((n,), -7.0, dtype=torch.float32, device="cuda")  # noqa: E731
    i32 = lambda: torch.full((n,), -7, dtype=torch.int32, device="cuda")  # noqa: E731
    twist = torch.zeros(n, dtype=torch.float64, device="cuda")
    out = [f32(), f32(), f32(), i32(), f32(), f32(), f32(), i32()] + [f32() for _ in range(5)]
    length = torch.zeros(n, dtype=torch.float64, device="cuda")
    dummy = torch.zeros(1, dtype=torch.float32, device="cuda")
    args = [flat(c) for c in b] + [t(b[0].shape, torch.int32)]
    args += ([flat(c) for c in cur] if cur is not None else [dummy] * 3)
    args += [twist if cur is not None else dummy, torch.tensor([cur is not None], device="cuda")]
    args += [t(p[:, i], torch.float32) for i in range(3)] + [t([0.0, 0.0, 1.0], torch.float32)] + out
    args += [t([0.25], torch.float32), t([n], torch.int64), length, t([0.01], torch.float32)]
    k = fq.kernels.compileTraceBlineScott()
    k.schedule = schedule
    k((28, 1), (128, 1, 1), tuple(args))
    torch.cuda.synchronize()
    return [a.cpu().numpy() for a in out + [length, twist]]


@pytest.mark.parametrize("shape,lines", [((32, 32, 32), 200), ((32, 32, 31), 200), ((33, 37, 41), 97), ((33, 37, 41), 98),
                                         ((2, 150, 120), 3000), ((150, 2, 120), 3000), ((130, 121, 2), 3000),
                                         ((61, 50, 43), 70001)])
@pytest.mark.parametrize("twist", [False, True])
def test_paired_field_gives_the_bits_of_the_field_in_place(shape, lines, twist):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import fastqsl_amd as fq
    b = [np.asarray(c, np.float32) for c in synth.multipole(shape, seed=5, count=10, device="cpu")]
    cur = [b[1], b[2], b[0]] if twist else None   # any field serves as the current
    rng = np.random.default_rng(2)
    p = (rng.uniform(-0.02, 1.02, (lines, 3)) * (np.array(shape) - 1)).astype(np.float32)
    p[: lines // 2, 2] = 0.0
    p[lines // 2: lines // 2 + 20] = np.round(p[lines // 2: lines // 2 + 20])
    p[3], p[5, 2], p[7] = np.nan, -0.5, np.array(shape) + 50.0
    ref = _call(torch, fq, b, cur, p, "per_line")
    for _ in range(2):
        got = _call(torch, fq, b, cur, p, "persistent")
        for k, (g, r) in enumerate(zip(got, ref)):
            np.testing.assert_array_equal(g, r, err_msg=str(k))
        fq.Field(*synth.multipole((64, 64, 60), seed=8, count=3, device="cpu")).close()
