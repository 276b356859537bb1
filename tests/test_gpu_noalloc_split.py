"""d_noFlagOCCSolver_noalloc where few unoccupied bands lie beside many
occupied ones: the direct form splits its G ranges there, whose partial sums
(kept per band, occupied ones too) must still fit the launcher's 16 MiB.
Bitwise equal to d_noFlagOCCSolver."""
import numpy as np
import pytest

import gpp_inputs
from test_zz_no_alloc import _device, _get, _launch, _outs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,nv,ncouls,ngpown", [
    (508, 500, 2000, 300),   # whole ranges take 3.7 MB, five of them 18
    (1200, 1196, 900, 500),  # 14.4 MB whole: no room for a second range
    (130, 2, 1500, 70),      # split within the limit
])
def test_noalloc_beside_many_occupied_bands(gpplib, nb, nv, ncouls, ngpown):
    a = gpp_inputs.seeded_inputs(nb, ncouls, ngpown, seed=nb)
    d = _device(a)
    o1, o2 = _outs(nb), _outs(nb)
    assert _launch(gpplib, "d_noFlagOCCSolver", a, d, nv, o1) == 0
    assert _launch(gpplib, "d_noFlagOCCSolver_noalloc", a, d, nv, o2) == 0, gpplib.gpp_last_error()
    for x, y in zip(_get(o1), _get(o2)):
        np.testing.assert_array_equal(x, y)
