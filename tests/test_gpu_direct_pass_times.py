"""Direct forms: what a pass of frequencies costs.  The device clock's stage
times of one shape at several frequency counts, least of several evaluations,
against each other."""
import pytest

import gpp_inputs
from test_gpu_parity import problem_of

pytestmark = pytest.mark.gpu


def stage_ms(ctx, arrs, nv, nf, form):
    arrs["wx_array"] = gpp_inputs.seeded_inputs(1, 4, 1, nfreq=nf, seed=0, dw=0.3)["wx_array"]
    ctx.upload(problem_of(arrs, nv), arrs)
    best = 1e9
    for _ in range(12):
        ctx.sigma(form)
        best = min(best, sum(v for k, v in ctx.last_timing().items() if k.startswith("direct_unoccupied")))
    return best


@pytest.mark.parametrize("form", ["direct", "direct-strict"])
def test_two_frequencies_cost_less_than_three(ctx, form):
    """A pass of two runs two thirds of the updates of one of three."""
    arrs = gpp_inputs.seeded_inputs(200, 3000, 150, seed=44)
    two, three = stage_ms(ctx, arrs, 3, 2, form), stage_ms(ctx, arrs, 3, 3, form)
    assert two < three, (two, three)


@pytest.mark.parametrize("form,few,many", [("direct", 5, 8), ("direct-strict", 4, 6), ("direct-strict", 5, 8)])
def test_a_narrow_last_pass_costs_less_than_a_whole_one(ctx, form, few, many):
    """The work is few / many of it (at most 0.67) and the pass count the same
    or less; 0.9 leaves room for what a pass costs whatever its width.  Wide and
    narrow passes dealt out unevenly over the XCDs cost what two wide ones do."""
    arrs = gpp_inputs.seeded_inputs(200, 3000, 150, seed=45)
    a, b = stage_ms(ctx, arrs, 3, few, form), stage_ms(ctx, arrs, 3, many, form)
    assert a < 0.9 * b, (a, b)


@pytest.mark.parametrize("form", ["direct", "direct-strict"])
def test_four_frequencies_are_one_pass(ctx, form):
    """A pass of four loads and reduces what one of three does, so it takes at
    most the time per update of one of three: 4 / 3 in all."""
    arrs = gpp_inputs.seeded_inputs(200, 3000, 150, seed=46)
    three, four = stage_ms(ctx, arrs, 3, 3, form), stage_ms(ctx, arrs, 3, 4, form)
    assert four < 4 / 3 * three, (three, four)
