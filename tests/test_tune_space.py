"""The autotuner searches the knobs that the request's launches read, and no others."""
import os
import re

import pytest

from fastqsl_amd import tune

SRC = open(os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fastqsl_amd", "csrc",
                        "fqsl_kernels.hip")).read()


@pytest.mark.parametrize("kw,lanes", [
    (dict(precision="fp32c", lines=1 << 22), False),
    (dict(precision="fp32c", method="rk4", lines=1 << 20), False),
    (dict(precision="fp32c", method="rk4", lines=(1 << 20) + 1), True),
    (dict(precision="fp64", lines=1000), False),
    (dict(precision="fp64", lines=70000), True),
    (dict(precision="mixed", lines=10), True),
])
def test_single_requests(kw, lanes):
    knobs = tune.searched(**kw)
    assert set(knobs) <= set(tune.SPACE) and "scott_waves" not in knobs
    assert {"order", "order_buckets", "grid_pct"} <= set(knobs)
    assert ("refill_min" in knobs) == ("queues" in knobs) == lanes


@pytest.mark.parametrize("precision,lines,expected", [
    ("fp32c", 1 << 23, {"grid_pct"}), ("fp32c", (1 << 23) + 1, {"grid_pct", "refill_min"}),
    ("fp64", 70000, {"grid_pct", "refill_min"}), ("mixed", 5, {"grid_pct", "refill_min"}),
])
def test_batches(precision, lines, expected):
    assert set(tune.searched(precision, lines=lines, batch=True)) == expected == set(tune.BATCH_SPACE) & expected


def test_the_search_measures_no_other_knob():
    seen = set()
    space = {k: tune.SPACE[k] for k in tune.searched("fp32c", lines=1 << 20)}

    def cost(cfg):
        seen.update(k for k, v in cfg.items() if v != tune.DEFAULTS[k])
        return 1.0

    best, _, _ = tune.coordinate_descent(cost, space=space)
    assert best == tune.DEFAULTS and seen == set(space)


def test_only_the_per_line_schedule_reads_the_wave_knob():
    reads = [m.start() for m in re.finditer(r"g_tune\[FQSL_TUNE_SCOTT_WAVES\]", SRC)]
    assert len(reads) == 1
    body = SRC[SRC.index("static int scott_waves("):]
    assert SRC.index("static int scott_waves(") < reads[0] < SRC.index("static int scott_waves(") + body.index("}")
    uses = [m.start() for m in re.finditer(r"scott_waves<", SRC)]
    assert len(uses) == 1 and "FQSL_SCHED_PER_LINE" in SRC[uses[0] - 400:uses[0]]
