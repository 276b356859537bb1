"""Memory of the products Mu where band groups hold several at a time."""
import ctypes

import numpy as np
import pytest

import hiprt

pytestmark = pytest.mark.gpu


def free_bytes():
    rt = hiprt.rt()
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert rt.hipDeviceSynchronize() == 0
    assert rt.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def rows(nb, groups, lo):
    k = np.arange(nb) % groups
    return lo + 0.7 * k[:, None] + np.array([0.0, 0.5, 1.0])[None, :]


@pytest.mark.parametrize("nv", [0, 5])
def test_fused_reduce_holds_one_product(gpplib, nv):
    """GPP_OPT_FUSED_REDUCE is for problems whose Mu does not fit: of ten
    groups the one that cannot be fused (a negative frequency, with five
    occupied bands all of them) needs its Mu, one at a time."""
    import pygpp
    nb, ncouls, ngpown = 40, 8192, 1024
    mu = 16 * ncouls * ngpown
    with pygpp.Context(0) as c:
        c.generate_seeded(pygpp.Problem(nb, nv, ncouls, ngpown, 3), 9)
        c.set_band_frequencies(rows(nb, 10, -0.2))
        assert c.band_buckets() == 10
        c.set_option(pygpp.GPP_OPT_FUSED_REDUCE, 1)
        before = free_bytes()
        c.sigma("factored-f64")
        assert c.last_form() == "factored-f64"
        # the rest: Bg and the permuted aqsn (6 MB), partial sums (10 MB)
        assert before - free_bytes() < 2 * mu
