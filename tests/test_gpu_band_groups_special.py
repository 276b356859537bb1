"""Band-dependent frequencies over values that are not finite or make terms that
are not: a frequency of one group exactly on a pole, infinities and NaN in each
input, a term that overflows.  What is finite in the oracle's per-band loop is
finite here, within the factored forms' 1e-10, and nothing else is."""
import numpy as np
import pytest

import gpp_inputs
from test_gpu_band_groups import KEYS, _rows
from test_gpu_parity import assert_close, problem_of

pytestmark = pytest.mark.gpu

NB, NV, NC, NG, GROUPS = 41, 3, 530, 21, 5


def place(a, kind, layout):
    """The element that differs, in the last column and G-vector or near."""
    band = NB - 1                       # in a group without occupied bands
    if kind == "pole":                  # frequency 1 of that band's group
        a["wtilde_array"][NG - 1, NC - 1] = a["wx_array"][band, 1]
    elif kind == "pole_occupied":
        a["wtilde_array"][2, 17] = a["wx_array"][0, 1]
    elif kind == "wtilde_inf":
        a["wtilde_array"][NG - 1, 256] = np.inf
    elif kind == "wtilde_overflow":
        a["wtilde_array"][NG - 1, 256] = 1e200
    elif kind == "wtilde_large":
        a["wtilde_array"][NG - 1, 256] = 1e100
    elif kind == "ieps_inf":
        a["I_eps_array"][0, NC - 1] = np.inf
    elif kind == "ieps_nan":
        a["I_eps_array"][NG - 1, 511] = np.nan
    elif kind == "aqsn_nan":
        a["aqsntemp"][band, NC - 1] = np.nan
    elif kind == "aqsn_nan_group_end":  # the last band of a group, beside the next one's first
        k = _rows(NB, NV, a["wx_array"].shape[1], GROUPS, layout)[:, 0]
        a["aqsntemp"][np.flatnonzero(k == k[NB // 2])[-1], 5] = np.nan


@pytest.mark.parametrize("nf", [3, 6])
@pytest.mark.parametrize("layout", ["together", "interleaved"])
@pytest.mark.parametrize("kind", ["pole", "pole_occupied", "wtilde_inf", "wtilde_overflow", "wtilde_large", "ieps_inf",
                                  "ieps_nan", "aqsn_nan", "aqsn_nan_group_end"])
def test_what_is_finite_stays_finite(ctx, oracle, kind, layout, nf):
    a = gpp_inputs.seeded_inputs(NB, NC, NG, nfreq=nf, seed=17)
    a["wx_array"] = 3.0 + _rows(NB, NV, nf, GROUPS, layout)
    place(a, kind, layout)
    ctx.upload(problem_of(a, NV), a)
    assert ctx.band_buckets() == GROUPS
    ref = oracle.sigma(a, nvband=NV, threads=4)
    out = ctx.sigma("factored-f64", acht_n1_loc=True)
    for k in KEYS:
        r, g = np.atleast_1d(ref[k]), np.atleast_1d(out[k])
        np.testing.assert_array_equal(np.isfinite(g), np.isfinite(r), err_msg=k)
        ok = np.isfinite(r)
        assert_close({k: g[ok]}, {k: r[ok]}, 1e-10, (k,)) if ok.any() else None
    assert (kind == "wtilde_large") == all(np.isfinite(ref[k]).all() for k in KEYS)
