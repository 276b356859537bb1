"""The FP64 Gram and acht products at the edges of their stages and tiles.  Every Gram tile gives
the same bits (each Mu entry is the same sum in the same order), within 1e-10
of the oracle.  Option 0 picks by size: the 16 x 16 tile for the first list, the
32 x 64 one for the second."""
import numpy as np
import pytest

import gpp_inputs
from test_gpu_factored import KEYS, TOL_FACTORED
from test_gpu_parity import assert_close, problem_of

pytestmark = pytest.mark.gpu

# nb, nv, ncouls, ngpown: bands against stages of 8 (64 x 128, 128 x 64: three
# buffers; 64 x 64: four) and 24 (16 x 16: six buffers)
SMALL = [
    (4, 4, 70, 5),       # no band: Mu is zero
    (3, 2, 100, 16),     # one band
    (9, 2, 129, 33),     # 7, 8, 9: around one stage of 8
    (10, 2, 128, 64),
    (11, 2, 127, 65),
    (18, 2, 16, 17),     # 16, 17
    (19, 2, 257, 31),
    (26, 2, 300, 32),    # 24, 25: three stages of 8, one of 24
    (27, 2, 333, 97),
    (34, 2, 65, 130),    # 32, 33
    (35, 2, 500, 40),
    (146, 2, 200, 15),   # 144, 145, 168, 169: the ring of 24 whole, one more, twice around
    (147, 2, 90, 48),
    (170, 2, 64, 49),
    (171, 2, 17, 1),
]
MIDDLE = [(100, 3, 4100, 130), (67, 2, 4096, 128)]


@pytest.mark.parametrize("shape", SMALL + MIDDLE, ids=lambda s: "x".join(map(str, s)))
def test_gram_tiles_at_their_edges(ctx, oracle, shape):
    import pygpp
    nb, nv, ncouls, ngpown = shape
    ngpown = min(ngpown, ncouls)
    arrs = gpp_inputs.seeded_inputs(nb, ncouls, ngpown, seed=sum(shape))
    ctx.upload(problem_of(arrs, nv), arrs)
    out = []
    try:
        for tile in range(4):
            ctx.set_option(pygpp.GPP_OPT_GRAM_TILE, tile)
            out.append(ctx.sigma("factored-f64"))
    finally:
        ctx.set_option(pygpp.GPP_OPT_GRAM_TILE, 0)
    assert_close(out[0], oracle.sigma(arrs, nvband=nv, threads=8), TOL_FACTORED, KEYS)
    for tile in range(1, 4):
        for k in KEYS:
            np.testing.assert_array_equal(out[tile][k], out[0][k], err_msg=f"tile {tile} {k}")


# nb, nv, ncouls, ngpown: G-vector stages of 8 against splits of at least 32,
# tiles of 64 rows (a last one of at most 32 runs half) by 128 or 64 bands
ACHT = [
    (4, 2, 7, 5),        # one partial stage
    (20, 3, 8, 8),
    (67, 2, 33, 32),     # 65 bands: the wider tile's edge
    (66, 2, 64, 33),     # 64 bands, 33 rows
    (131, 3, 257, 65),   # 128 bands, a last tile of one row
    (60, 0, 1000, 96),
    (200, 8, 2100, 97),  # occupied bands by their own launch
    (300, 3, 4100, 130),
]


@pytest.mark.parametrize("shape", ACHT, ids=lambda s: "x".join(map(str, s)))
def test_acht_product_at_its_edges(ctx, oracle, shape):
    """acht_n1_loc of the factored form against the oracle, bitwise repeatable."""
    nb, nv, ncouls, ngpown = shape
    arrs = gpp_inputs.seeded_inputs(nb, ncouls, min(ngpown, ncouls), seed=sum(shape) + 1)
    ctx.upload(problem_of(arrs, nv), arrs)
    out = ctx.sigma("factored-f64", acht_n1_loc=True)
    assert_close(out, oracle.sigma(arrs, nvband=nv, threads=8), TOL_FACTORED, KEYS + ("acht_n1_loc",))
    again = ctx.sigma("factored-f64", acht_n1_loc=True)
    np.testing.assert_array_equal(out["acht_n1_loc"], again["acht_n1_loc"])
