"""The product kernels that no option selects, at the edges of their stages and
tiles, at shapes for which the size rules pick them (tests/test_tile_choice.py).
Mu is the same sum in the same order in every Gram tile: the same bits, within
1e-10 of the oracle."""
import numpy as np
import pytest

import gpp_inputs
from test_gpu_factored import KEYS, TOL_FACTORED
from test_gpu_parity import assert_close, problem_of
from test_tile_choice import ACHT_128, ACHT_128_CUT, GRAM_16, GRAM_32, GROUPS_16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", GRAM_16 + GRAM_32, ids=lambda s: "x".join(map(str, s)))
def test_gram_tiles_chosen_by_size(ctx, oracle, shape):
    import pygpp
    nb, nv, ncouls, ngpown = shape
    rng = np.random.default_rng(sum(shape))
    a = gpp_inputs.seeded_inputs(nb, ncouls, min(ngpown, ncouls), seed=sum(shape))
    if ngpown > ncouls:  # columns of the same distributions, indices repeated
        for k in ("I_eps_array", "wtilde_array"):
            a[k] = a[k][rng.integers(0, ncouls, ngpown)] * (1 + 0.01 * rng.random((ngpown, 1)))
        a["inv_igp_index"] = np.sort(rng.integers(0, ncouls, ngpown)).astype(np.int32)
    ctx.upload(problem_of(a, nv), a)
    assert ctx.problem.ngpown == ngpown
    out = ctx.sigma("factored-f64")
    assert_close(out, oracle.sigma(a, nvband=nv, threads=8), TOL_FACTORED, KEYS)
    try:
        for tile in (1, 2, 3):
            ctx.set_option(pygpp.GPP_OPT_GRAM_TILE, tile)
            same = ctx.sigma("factored-f64")
            for k in KEYS:
                np.testing.assert_array_equal(same[k], out[k], err_msg=f"tile {tile} {k}")
    finally:
        ctx.set_option(pygpp.GPP_OPT_GRAM_TILE, 0)


@pytest.mark.parametrize("nf", [2, 5])
def test_groups_of_few_bands_in_one_launch(ctx, oracle, nf):
    """16 x 16 tiles over groups without an unoccupied band, with one, and with
    one stage and a band more or less."""
    import pygpp
    nv, un = GROUPS_16["nv"], GROUPS_16["unoccupied"]
    k = np.concatenate([np.zeros(nv, int)] + [np.full(n, i) for i, n in enumerate(un)])
    nb = len(k)
    a = gpp_inputs.seeded_inputs(nb, GROUPS_16["ncouls"], GROUPS_16["ngpown"], nfreq=nf, seed=91)
    a["wx_array"] = 7.0 + 0.9 * k[:, None] + 0.5 * np.arange(nf)[None, :]
    ctx.upload(problem_of(a, nv), a)
    assert ctx.band_buckets() == len(un)
    out = ctx.sigma("factored-f64", acht_n1_loc=True)
    assert_close(out, oracle.sigma(a, nvband=nv, threads=8), TOL_FACTORED, KEYS + ("acht_n1_loc",))
    try:
        for tile in (1, 2, 3):
            ctx.set_option(pygpp.GPP_OPT_GRAM_TILE, tile)
            same = ctx.sigma("factored-f64")
            for key in KEYS:
                np.testing.assert_array_equal(same[key], out[key], err_msg=f"tile {tile} {key}")
    finally:
        ctx.set_option(pygpp.GPP_OPT_GRAM_TILE, 0)


@pytest.mark.parametrize("shape", ACHT_128_CUT + ACHT_128, ids=lambda s: "x".join(map(str, s)))
def test_acht_tiles_chosen_by_size(ctx, oracle, shape):
    nb, nv, ncouls, ngpown = shape
    a = gpp_inputs.seeded_inputs(nb, ncouls, ngpown, seed=sum(shape) + 1)
    ctx.upload(problem_of(a, nv), a)
    out = ctx.sigma("factored-f64", acht_n1_loc=True)
    assert_close(out, oracle.sigma(a, nvband=nv, threads=8), TOL_FACTORED, KEYS + ("acht_n1_loc",))
    again = ctx.sigma("factored-f64", acht_n1_loc=True)
    np.testing.assert_array_equal(out["acht_n1_loc"], again["acht_n1_loc"])
