"""The direct forms where their launch changes shape: G ranges split and whole,
ranges of uneven chunks, frequency passes with every remainder, column tiles and
band groups with one live entry, occupied bands only -- against the oracle."""
import numpy as np
import pytest

import gpp_inputs
from test_gpu_parity import TOL, assert_close, problem_of

pytestmark = pytest.mark.gpu

# nb, nv, ncouls, ngpown, nfreq
SHAPES = [
    (10, 1, 63, 1, 1),        # one partial chunk
    (11, 2, 65, 5, 2),        # one live column in the last tile
    (19, 2, 385, 9, 3),       # seven chunks: one range
    (19, 3, 833, 9, 4),       # fourteen: two uneven ranges
    (18, 2, 1664, 13, 5),     # passes 4 + 1 (strict 3 + 2)
    (33, 4, 2500, 12, 6),
    (9, 8, 3000, 17, 7),      # one unoccupied band
    (24, 0, 1999, 8, 9),      # no occupied band
    (3, 3, 6500, 5, 3),       # no unoccupied band, many ranges
    (512, 2, 800, 40, 3),     # a split by the blocks in flight
]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("form", ["direct", "direct-strict"])
def test_direct_split_vs_oracle(ctx, oracle, form, shape):
    nb, nv, ncouls, ngpown, nfreq = shape
    arrs = gpp_inputs.seeded_inputs(nb, ncouls, ngpown, nfreq=nfreq, seed=sum(shape), dw=0.3)
    ctx.upload(problem_of(arrs, nv), arrs)
    out = ctx.sigma(form)
    assert_close(out, oracle.sigma(arrs, nvband=nv, threads=8), TOL)
    again = ctx.sigma(form)
    for k in out:
        np.testing.assert_array_equal(out[k], again[k], err_msg=k)


def test_launchers_leave_outputs_alone_on_a_bad_index(ctx, gpplib):
    """A negative index is reported by every launcher, with nothing added; the
    next call on good indices adds its results."""
    import hiprt
    import pygpp
    nb, nv, ncouls, ngpown = 20, 3, 900, 21
    arrs = gpp_inputs.seeded_inputs(nb, ncouls, ngpown, seed=8)
    ctx.upload(problem_of(arrs, nv), arrs)
    want = ctx.sigma("direct")
    bad = dict(arrs, inv_igp_index=arrs["inv_igp_index"].copy())
    bad["inv_igp_index"][ngpown - 1] = -1
    re, im, n1loc = (hiprt.DeviceArray(np.zeros(n, t)) for n, t in
                     ((3, np.float64), (3, np.float64), (nb, np.complex128)))
    asx, sre, sim = (hiprt.DeviceArray(np.zeros(n, t)) for n, t in
                     ((3, np.complex128), (1, np.float64), (1, np.float64)))

    def launch(a):
        d = {k: hiprt.DeviceArray(v) for k, v in a.items()}
        p = {k: v.ptr for k, v in d.items()}
        st = [gpplib.d_reduce_achstemp(nb, p["inv_igp_index"], ncouls, p["aqsmtemp"], p["aqsntemp"],
                                       p["I_eps_array"], sre.ptr, sim.ptr, ngpown, p["vcoul"]),
              gpplib.d_till_nvband(nv, ngpown, ncouls, p["inv_igp_index"], p["wx_array"], p["wtilde_array"],
                                   p["aqsmtemp"], p["aqsntemp"], p["I_eps_array"], asx.ptr, p["vcoul"], n1loc.ptr,
                                   re.ptr, im.ptr, 1.0),
              gpplib.d_noFlagOCCSolver(nb, nv, ngpown, ncouls, p["inv_igp_index"], p["wx_array"], p["wtilde_array"],
                                       p["aqsmtemp"], p["aqsntemp"], p["I_eps_array"], p["vcoul"], re.ptr, im.ptr,
                                       n1loc.ptr)]
        got = {"achtemp": re.get() + 1j * im.get(), "asxtemp": asx.get(), "acht_n1_loc": n1loc.get(),
               "achstemp": sre.get()[0] + 1j * sim.get()[0]}
        return st, got

    st, got = launch(bad)
    assert st == [pygpp.GPP_ERR_BAD_INDEX] * 3
    assert all(not np.any(v) for v in got.values())
    st, got = launch(arrs)
    assert st == [pygpp.GPP_OK] * 3
    assert_close(got, want, tol=1e-13)
