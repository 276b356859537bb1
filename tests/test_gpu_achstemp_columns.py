"""achstemp where its launches change with the number of columns: entries formed
by the waves that use them or in a launch before (3072 columns), the launcher's
own kernel or the factored forms' (1024) -- against the oracle, and the gathered
rows through the outputs that need them."""
import numpy as np
import pytest

import gpp_inputs
import hiprt
from test_gpu_factored import TOL_FACTORED
from test_gpu_parity import TOL, assert_close, problem_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ngpown", [1023, 1024, 3071, 3072, 3300])
def test_achstemp_columns(ctx, gpplib, oracle, ngpown):
    nb, nv, ncouls = 5, 2, 400
    rng = np.random.default_rng(ngpown)
    a = gpp_inputs.seeded_inputs(nb, ncouls, 1, seed=ngpown)
    a["inv_igp_index"] = rng.integers(0, ncouls, ngpown).astype(np.int32)
    a["I_eps_array"] = rng.uniform(-0.5, 0.5, (ngpown, ncouls)) + 1j * rng.uniform(-0.5, 0.5, (ngpown, ncouls))
    a["wtilde_array"] = rng.uniform(0.5, 5, (ngpown, ncouls)) + 1j * rng.uniform(-0.05, 0.05, (ngpown, ncouls))
    a["I_eps_array"][::7] = 1e-7  # below the threshold of gppComplex.cpp:91
    ref = oracle.sigma(a, nvband=nv, threads=8)
    ctx.upload(problem_of(a, nv), a)
    assert_close(ctx.sigma("factored-f64"), ref, TOL_FACTORED, ("achtemp", "asxtemp"))
    assert_close(ctx.sigma("factored-f64"), ref, TOL, ("achstemp",))
    assert_close(ctx.sigma("direct"), ref, TOL, ("achstemp",))
    d = {k: hiprt.DeviceArray(v) for k, v in a.items()}
    re, im = hiprt.DeviceArray(np.zeros(1)), hiprt.DeviceArray(np.zeros(1))
    assert gpplib.d_reduce_achstemp(nb, d["inv_igp_index"].ptr, ncouls, d["aqsmtemp"].ptr, d["aqsntemp"].ptr,
                                    d["I_eps_array"].ptr, re.ptr, im.ptr, ngpown, d["vcoul"].ptr) == 0
    assert_close({"achstemp": re.get()[0] + 1j * im.get()[0]}, ref, TOL, ("achstemp",))
