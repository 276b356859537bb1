"""The direct forms with more blocks than one grid dimension takes (512 threads
each: 2^32 threads are 8388608 blocks): many bands and columns over few
G-vectors.  The whole against the sum of its two halves of the columns, which
one dimension takes.  All terms are positive, so a component is a sum of at
most about 200 rounded additions deep (128 partials a lane, 33 bands a thread,
trees): 200 eps, 4.4e-14, bounds the difference of the two orders."""
import numpy as np
import pytest

from test_gpu_parity import problem_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["direct", "direct-strict"])
def test_more_blocks_than_one_dimension(ctx, form):
    nb, nv, ncouls, ngpown = 8200, 2, 4, 32768
    assert (nb - nv + 7) // 8 * (ngpown // 4) * 512 > 2 ** 32
    rng = np.random.default_rng(7)

    def real(shape, lo, hi):
        return rng.uniform(lo, hi, shape) + 0j

    a = {"inv_igp_index": rng.integers(0, ncouls, ngpown).astype(np.int32), "wx_array": np.array([10.0]),
         "vcoul": rng.uniform(0.1, 10.0, ncouls), "aqsmtemp": real((nb, ncouls), 0.5, 1), "aqsntemp": real((nb, ncouls), 0.5, 1),
         "I_eps_array": real((ngpown, ncouls), 0.1, 0.5), "wtilde_array": real((ngpown, ncouls), 0.5, 5)}
    ctx.upload(problem_of(a, nv), a)
    whole = ctx.sigma(form)
    halves = []
    for j in (0, ngpown // 2):
        ctx.set_columns(j, j + ngpown // 2)
        halves.append(ctx.sigma(form))
    ctx.set_columns(0, 0)
    for k in ("achtemp", "asxtemp", "acht_n1_loc", "achstemp"):
        want = np.asarray(halves[0][k]) + halves[1][k]
        assert np.all(np.real(want) != 0)
        np.testing.assert_allclose(whole[k], want, rtol=4.4e-14, atol=0, err_msg=k)
