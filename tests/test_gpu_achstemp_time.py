"""d_reduce_achstemp with many columns costs what the factored forms' gather
stage does, which forms the same sums and stores the gathered rows besides."""
import time

import numpy as np
import pytest

import gpp_inputs
import hiprt
from test_gpu_parity import problem_of

pytestmark = pytest.mark.gpu


def launcher_us(lib, d, nb, ncouls, ngpown, out):
    best = 1e9
    for _ in range(30):
        t0 = time.perf_counter()
        assert lib.d_reduce_achstemp(nb, d["inv_igp_index"].ptr, ncouls, d["aqsmtemp"].ptr, d["aqsntemp"].ptr,
                                     d["I_eps_array"].ptr, out[0].ptr, out[1].ptr, ngpown, d["vcoul"].ptr) == 0
        assert hiprt.rt().hipDeviceSynchronize() == 0
        best = min(best, 1e6 * (time.perf_counter() - t0))
    return best


def test_many_columns_cost_what_the_gather_stage_does(ctx, gpplib):
    """The rest of a launcher's call (check, launches, wait) is what it takes
    on one column; half as much again as the stage is the margin."""
    nb, ncouls, ngpown = 24, 512, 20000
    rng = np.random.default_rng(3)
    a = gpp_inputs.seeded_inputs(nb, ncouls, 1, seed=3)
    a["inv_igp_index"] = rng.integers(0, ncouls, ngpown).astype(np.int32)
    a["I_eps_array"] = a["wtilde_array"] = rng.uniform(0.5, 1, (ngpown, ncouls)) + 0j
    d = {k: hiprt.DeviceArray(v) for k, v in a.items()}
    out = [hiprt.DeviceArray(np.zeros(1)) for _ in range(2)]
    whole, call = launcher_us(gpplib, d, nb, ncouls, ngpown, out), launcher_us(gpplib, d, nb, ncouls, 1, out)
    ctx.upload(problem_of(a, 2), a)
    stage = 1e9
    for _ in range(8):
        ctx.sigma("factored-f64")
        stage = min(stage, 1e3 * ctx.last_timing()["factored_gather_achstemp"])
    assert whole - call < 1.5 * stage, (whole, call, stage)
