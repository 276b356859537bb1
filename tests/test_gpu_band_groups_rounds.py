"""Band-dependent frequencies with more groups than are held at a time: the
products of one, two or three groups per round, rounds that hold groups with
occupied bands, groups without, and both, a last round that is not full -- with
and without acht_n1_loc, against the oracle's per-band loop at the factored
forms' 1e-10 per component, and at the size where the default 4 GB end."""
import ctypes

import numpy as np
import pytest

import gpp_inputs
from test_gpu_band_groups import KEYS, _rows
from test_gpu_parity import assert_close, problem_of

pytestmark = pytest.mark.gpu

DEFAULT = 4 << 30


def hold(lib, ctx, nbytes):
    """Bytes of Mu that an evaluation holds at a time."""
    lib.gpp_test_bucket_mu.argtypes = [ctypes.c_void_p, ctypes.c_size_t]
    lib.gpp_test_bucket_mu.restype = None
    lib.gpp_test_bucket_mu(ctx._h, nbytes)


@pytest.mark.parametrize("form,nb,nv,nc,ng,nf,groups,layout", [
    ("factored-f64", 33, 2, 1023, 17, 3, 7, "together"),      # one occupied group, six bare
    ("factored-f64", 40, 3, 1025, 33, 2, 7, "interleaved"),   # three occupied, four bare
    ("factored-f64", 40, 0, 700, 20, 5, 5, "interleaved"),    # all bare
    ("factored-f64", 20, 17, 520, 9, 9, 5, "interleaved"),    # all occupied
    ("factored-f64", 37, 5, 2049, 70, 3, 4, "single"),
    ("factored-ozaki-i8", 40, 4, 700, 30, 3, 5, "interleaved"),
    ("factored-ozaki", 30, 2, 300, 21, 4, 4, "together"),
])
def test_rounds_vs_oracle(ctx, gpplib, oracle, form, nb, nv, nc, ng, nf, groups, layout):
    a = gpp_inputs.seeded_inputs(nb, nc, ng, nfreq=nf, seed=nb + nc + 1)
    a["wx_array"] = _rows(nb, nv, nf, groups, layout)
    ctx.upload(problem_of(a, nv), a)
    assert ctx.band_buckets() == groups
    ref = oracle.sigma(a, nvband=nv, threads=8)
    mu = 16 * nc * ng
    try:
        for per_round in (0, 1, 2, 3, groups - 1, groups):
            hold(gpplib, ctx, per_round * mu + 8)
            out = ctx.sigma(form, acht_n1_loc=True)
            assert ctx.last_form() == form
            assert_close(out, ref, 1e-10, KEYS)
            plain = ctx.sigma(form)
            for k in ("achtemp", "asxtemp", "achstemp"):
                np.testing.assert_array_equal(plain[k], out[k], err_msg=f"{per_round} {k}")
    finally:
        hold(gpplib, ctx, DEFAULT)


def test_rounds_at_the_default_limit(ctx, gpplib, oracle):
    """Eleven groups of 859 MB: rounds of five, five and one."""
    import pygpp
    nb, nv, groups = 24, 2, 11
    p = pygpp.Problem(nb, nv, 32768, 1638, 2)
    assert DEFAULT // (16 * 32768 * 1638) == 5
    a = pygpp.fill_seeded(p, seed=6)
    a["wx_array"] = _rows(nb, nv, 2, groups, "interleaved")
    ctx.upload(p, a)
    assert ctx.band_buckets() == groups
    assert_close(ctx.sigma("factored-f64", acht_n1_loc=True), oracle.sigma(a, nvband=nv, threads=16), 1e-10, KEYS)
