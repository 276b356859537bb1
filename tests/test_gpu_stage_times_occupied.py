"""Stage times where the two occupied bands are all there are: their
acht_n1_loc terms are summed by the pole reduce, so that the stage's only
launch is the final sum, which has to note the stage's start."""
import pytest

import gpp_inputs
from test_gpu_parity import problem_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nfreq", [3, 5])
@pytest.mark.parametrize("form", ["factored-f64", "factored-ozaki", "factored-ozaki-i8"])
def test_stage_times_two_occupied_bands(ctx, form, nfreq):
    arrs = gpp_inputs.seeded_inputs(2, 300, 20, nfreq=nfreq, seed=31)
    ctx.upload(problem_of(arrs, 2), arrs)
    for _ in range(2):
        ctx.sigma(form, acht_n1_loc=True)
        t = ctx.last_timing()
        total = t.pop("total")
        assert "factored_acht" in t and all(0 < v < 1e3 for v in t.values()), t
        assert abs(sum(t.values()) - total) < 1e-9
