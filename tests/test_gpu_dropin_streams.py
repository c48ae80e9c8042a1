"""Reference-shaped Scott calls that pair their field's nodes, over streams.

Such a call returns before its trace has ended, so that one thread keeps several
streams busy; the pairs' memory passes on only when the trace that reads it is
done: calls on other fields, and a field built in between, do not disturb it.
"""
import numpy as np
import pytest

from fastqsl_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _prepare(torch, shape, lines, seed, tol):
    b = synth.multipole(shape, seed=seed, count=10, device="cpu")
    p = np.random.default_rng(seed).uniform(0.02, 0.98, (lines, 3)) * (np.array(shape) - 1)
    t = lambda a, dt: torch.as_tensor(np.ascontiguousarray(a), dtype=dt, device="cuda")  # noqa: E731
    f32 = lambda: torch.full((lines,), -7.0, dtype=torch.float32, device="cuda")  # noqa: E731
    i32 = lambda: torch.full((lines,), -7, dtype=torch.int32, device="cuda")  # noqa: E731
    out = [f32(), f32(), f32(), i32(), f32(), f32(), f32(), i32()] + [f32() for _ in range(5)]
    length, dummy = torch.zeros(lines, dtype=torch.float64, device="cuda"), torch.zeros(1, device="cuda")
    args = [t(np.asarray(c, np.float32).ravel(order="F"), torch.float32) for c in b] + [t(b[0].shape, torch.int32)]
    args += [dummy] * 4 + [torch.tensor([False], device="cuda")]
    args += [t(p[:, i], torch.float32) for i in range(3)] + [t([0.0, 0.0, 1.0], torch.float32)] + out
    args += [t([0.25], torch.float32), t([lines], torch.int64), length, t([tol], torch.float32)]
    torch.cuda.synchronize()
    return tuple(args), out + [length]


def test_overlapping_calls_give_their_own_results(torch):
    import fastqsl_amd as fq
    shape, lines = (80, 72, 64), 20000
    calls = [_prepare(torch, shape, lines, seed, 0.01) for seed in range(6)]
    kern = [fq.kernels.compileTraceBlineScott() for _ in calls]
    alone = []
    for k, (args, out) in zip(kern, calls):
        k((28, 1), (128, 1, 1), args)
        torch.cuda.synchronize()
        alone.append([a.cpu().numpy().copy() for a in out])
    streams = [torch.cuda.Stream() for _ in range(3)]
    for turn in range(3):
        for _, out in calls:
            for a in out:
                a.fill_(-7)
        torch.cuda.synchronize()
        for j, (k, (args, _)) in enumerate(zip(kern, calls)):
            with torch.cuda.stream(streams[(j + turn) % 3]):
                k((28, 1), (128, 1, 1), args)
            if j == 3:   # a field that wants a block of the pairs' size: 32 bytes a node
                n = shape[0] * shape[1] * shape[2] * 4
                fq.Field(*synth.multipole((n // 4096, 64, 64), seed=9, count=1, device="cpu"), layouts=("soa64",)).close()
        torch.cuda.synchronize()
        for j, ((_, out), ref) in enumerate(zip(calls, alone)):
            for q, (a, r) in enumerate(zip(out, ref)):
                np.testing.assert_array_equal(a.cpu().numpy(), r, err_msg=f"turn {turn}, call {j}, output {q}")


def test_the_call_returns_before_its_trace_ends(torch):
    import fastqsl_amd as fq
    args, out = _prepare(torch, (96, 96, 96), 1 << 20, 1, 1e-3)
    kern = fq.kernels.compileTraceBlineScott()
    kern((28, 1), (128, 1, 1), args)      # kernels loaded, memory there
    torch.cuda.synchronize()
    kern((28, 1), (128, 1, 1), args)
    assert not torch.cuda.current_stream().query()
    torch.cuda.synchronize()
    assert int((out[3] > 0).sum()) > 0
