"""Band-dependent frequencies over several groups in one evaluation: every
group's product in one launch, the groups without occupied bands in one reduce
over all of them, acht_n1_loc group by group.  Column and G-vector counts at
the edges of their blocks (4 elements a thread, 256 threads: 1024), frequency
counts at each pass width and over two passes, bands whose groups lie together
(nothing is permuted), interleaved, and with occupied bands in several groups.
Compared with the oracle's per-band loop; the bound is the factored forms'
1e-10 per component (tests/test_gpu_band_wx.py)."""
import numpy as np
import pytest

import gpp_inputs
from test_gpu_parity import assert_close, problem_of

pytestmark = pytest.mark.gpu

KEYS = ("achtemp", "asxtemp", "acht_n1_loc", "achstemp")


def _rows(nb, nv, nf, groups, layout):
    """Frequency row per band: `groups` energies, none at a pole of the inputs'."""
    if layout == "together":        # groups in band order, the occupied bands in the first
        k = np.where(np.arange(nb) < nv, 0, np.arange(nb) * groups // nb)
    elif layout == "interleaved":   # occupied bands in several groups
        k = np.arange(nb) % groups
    else:                           # one band a group, the rest in the first
        k = np.where(np.arange(nb) >= nb - groups + 1, np.arange(nb) - (nb - groups), 0)
    return 4.0 - 1.37 * k[:, None] + 0.5 * (np.arange(nf) - 0.5 * (nf - 1))[None, :]


@pytest.mark.parametrize("form,nb,nv,nc,ng,nf,groups,layout", [
    ("factored-f64", 24, 0, 1, 1, 1, 3, "together"),
    ("factored-f64", 33, 2, 1023, 17, 2, 4, "together"),
    ("factored-f64", 40, 2, 1025, 33, 3, 5, "interleaved"),
    ("factored-f64", 40, 0, 1024, 65, 4, 7, "interleaved"),
    ("factored-f64", 37, 5, 2049, 129, 6, 3, "single"),
    ("factored-f64", 61, 8, 700, 40, 8, 6, "together"),
    ("factored-f64", 30, 3, 650, 21, 13, 8, "interleaved"),
    ("factored-f64", 20, 17, 520, 9, 19, 4, "interleaved"),
    ("factored-ozaki", 40, 4, 700, 70, 5, 4, "interleaved"),
    ("factored-ozaki-i8", 40, 4, 700, 70, 3, 4, "together"),
])
def test_groups_vs_oracle(ctx, oracle, form, nb, nv, nc, ng, nf, groups, layout):
    a = gpp_inputs.seeded_inputs(nb, nc, ng, nfreq=nf, seed=nb + nc)
    a["wx_array"] = _rows(nb, nv, nf, groups, layout)
    ctx.upload(problem_of(a, nv), a)
    assert ctx.band_buckets() == groups
    ref = oracle.sigma(a, nvband=nv, threads=8)
    out = ctx.sigma(form, acht_n1_loc=True)
    assert ctx.last_form() == form
    assert_close(out, ref, 1e-10, KEYS)
    # the other outputs do not depend on whether acht_n1_loc is requested
    plain = ctx.sigma(form)
    for k in ("achtemp", "asxtemp", "achstemp"):
        np.testing.assert_array_equal(plain[k], out[k])


@pytest.mark.parametrize("nf", [2, 5])
def test_groups_fused(ctx, oracle, nf):
    """With the fused reduce: at most 3 frequencies in the product's epilogue
    (a group with a negative frequency on its own product and reduce), more of
    them on a product and reduce per group."""
    import pygpp
    a = gpp_inputs.seeded_inputs(40, 600, 35, nfreq=nf, seed=77)
    a["wx_array"] = _rows(40, 3, nf, 5, "interleaved")
    assert (a["wx_array"] < 0).any() and (a["wx_array"][0] > 0).all()
    ctx.upload(problem_of(a, 3), a)
    ref = oracle.sigma(a, nvband=3, threads=8)
    try:
        ctx.set_option(pygpp.GPP_OPT_FUSED_REDUCE, 1)
        out = ctx.sigma("factored-f64")
    finally:
        ctx.set_option(pygpp.GPP_OPT_FUSED_REDUCE, 0)
    assert_close(out, ref, 1e-10, ("achtemp", "asxtemp", "achstemp"))
