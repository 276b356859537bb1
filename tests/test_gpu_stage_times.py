"""Stage times noted by the launches themselves: every stage an evaluation runs
is positive, they add up to the total, and the total fits the host's clock --
also with no occupied or no unoccupied band, with acht_n1_loc, per-band
frequencies and more evaluations in flight than the ring keeps."""
import time

import numpy as np
import pytest

import gpp_inputs
from test_gpu_parity import problem_of

pytestmark = pytest.mark.gpu

SHAPES = [(24, 2, 1000, 50), (9, 0, 130, 9), (5, 5, 200, 6), (30, 3, 700, 40)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("form", ["direct", "direct-strict", "factored-f64", "factored-ozaki-i8"])
def test_stage_times(ctx, form, shape):
    nb, nv, ncouls, ngpown = shape
    arrs = gpp_inputs.seeded_inputs(nb, ncouls, ngpown, seed=sum(shape))
    ctx.upload(problem_of(arrs, nv), arrs)
    for acht in (False, True):
        ctx.sigma(form, acht_n1_loc=acht)
        t0 = time.perf_counter()
        ctx.sigma(form, acht_n1_loc=acht)
        host_ms = 1e3 * (time.perf_counter() - t0)
        t = ctx.last_timing()
        total = t.pop("total")
        assert all(v > 0 for v in t.values()), t
        assert abs(sum(t.values()) - total) < 1e-9 and total < host_ms
    for _ in range(40):
        ctx.sigma_async(form)
    ctx.wait()
    s = ctx.timing_summary(32)
    assert s["evaluations"] == 32 and 0 < s["total"] < 40


def test_stage_times_band_rows(ctx):
    arrs = gpp_inputs.seeded_inputs(30, 700, 40, seed=3)
    ctx.upload(problem_of(arrs, 3), arrs)
    ctx.set_band_frequencies(np.repeat(np.arange(3.0), 10)[:, None] + np.array([3.0, 4.0, 5.0]))
    ctx.sigma("factored-f64")
    t = ctx.last_timing()
    total = t.pop("total")
    assert t and all(v > 0 for v in t.values()) and abs(sum(t.values()) - total) < 1e-9
