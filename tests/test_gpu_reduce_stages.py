"""The pole reduce with four or more frequencies loads the occupied bands' rows
of a block's next 256 G-vectors through LDS: occupied band counts with a
kernel of their own (one to eight) and the general one's, G-vector counts at the edges of the 256, frequency counts at odd
groups of two and over several passes.  Against the oracle at the factored
forms' 1e-10 per component (tests/test_gpu_factored.py)."""
import pytest

import gpp_inputs
from test_gpu_parity import assert_close, problem_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nv,nc,nf", [
    (0, 257, 4), (1, 255, 5), (2, 256, 4), (2, 1023, 7), (3, 257, 8), (4, 513, 16), (5, 1, 4), (7, 300, 13),
    (8, 769, 9), (8, 512, 24), (9, 257, 16), (12, 511, 6), (1, 300, 3), (3, 257, 2), (5, 511, 3), (6, 770, 1),
    (6, 257, 20), (7, 255, 3),
])
def test_reduce_stages_vs_oracle(ctx, oracle, nv, nc, nf):
    ng = min(nc, 19)
    a = gpp_inputs.seeded_inputs(nv + 14, nc, ng, nfreq=nf, seed=900 + nv + nf)
    ctx.upload(problem_of(a, nv), a)
    out = ctx.sigma("factored-f64", acht_n1_loc=True)
    assert_close(out, oracle.sigma(a, nvband=nv, threads=8), 1e-10)
