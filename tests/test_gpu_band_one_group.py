"""Band-dependent frequencies that are one row for every band: the result is
the one of uploading that row, bit for bit, whatever the signs of the row
uploaded before it -- the ssx cutoff (gppComplex.cpp:58-59) is live at the
negative frequencies of the row that is evaluated."""
import numpy as np
import pytest

import gpp_inputs
from test_gpu_parity import problem_of

pytestmark = pytest.mark.gpu

FORMS = ["direct", "direct-strict", "factored-f64", "factored-ozaki-i8", "factored-ozaki"]


@pytest.mark.parametrize("fuse", [0, 1])
@pytest.mark.parametrize("nv", [2, 4])
@pytest.mark.parametrize("first,row", [([1.0, 2.0, 3.0], [-0.6, -0.2, 3.0]), ([-0.6, -0.2, 3.0], [1.0, 2.0, 3.0])],
                         ids=["positive_then_negative", "negative_then_positive"])
def test_one_group_is_the_row_whatever_its_signs(ctx, first, row, nv, fuse):
    import pygpp
    a = gpp_inputs.ssx_cutoff_inputs(14, 900, 40, seed=61)
    a.pop("_kind")
    try:
        ctx.set_option(pygpp.GPP_OPT_FUSED_REDUCE, fuse)
        for form in FORMS:
            for acht in (False, True):
                a["wx_array"] = np.array(row)
                ctx.upload(problem_of(a, nv), a)
                want = ctx.sigma(form, acht_n1_loc=acht)
                want_stages = set(ctx.last_timing())
                a["wx_array"] = np.array(first)
                ctx.upload(problem_of(a, nv), a)
                ctx.set_band_frequencies(np.tile(row, (14, 1)))
                assert ctx.band_buckets() == 1
                got = ctx.sigma(form, acht_n1_loc=acht)
                assert set(ctx.last_timing()) == want_stages, (form, acht)
                for k, v in want.items():
                    if v is not None:
                        np.testing.assert_array_equal(got[k], v, err_msg=f"{form} acht {acht} {k}")
    finally:
        ctx.set_option(pygpp.GPP_OPT_FUSED_REDUCE, 0)
