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


def test_groups_that_do_not_fit_together(gpplib):
    """Eighty groups of 4.3 GB asked for at once (344 GB) cannot be held: the
    evaluation runs with one at a time, bit for bit as when asked so, and keeps
    to it; nothing of the failed allocation is reported later."""
    import pygpp
    from test_gpu_band_groups_rounds import hold
    nb = 80
    with pygpp.Context(0) as c:
        c.generate_seeded(pygpp.Problem(nb, 2, 65536, 4096, 1), 10)
        c.set_option(pygpp.GPP_OPT_MAX_BUCKETS, nb)
        c.set_band_frequencies(3.0 + 0.01 * np.arange(nb)[:, None])
        hold(gpplib, c, 0)
        want = c.sigma("factored-f64")
        hold(gpplib, c, 1 << 40)
        for _ in range(2):
            got = c.sigma("factored-f64")
            assert c.last_form() == "factored-f64"
            for k in ("achtemp", "asxtemp", "achstemp"):
                np.testing.assert_array_equal(got[k], want[k])
