"""The 2D structure function with a general power and few lags, on both sides of
the line from which it sweeps columns (6144 blocks of grids wider than 128, three
lags and more), against the oracle.  Terms are non-negative: the bound on a sum's
relative error is that of test_gpu_structure_routes.py."""
import numpy as np
import pytest

from alsvinn_amd import BatchRunner
from tests.cases import smooth_state

pytestmark = pytest.mark.gpu

CASES = [
    # n, samples, number_of_h; a sample of 256 x 256 is 64 blocks a lag
    ((256, 256), 32, 4),   # 6144 blocks: swept
    ((256, 256), 31, 4),   # 5952
    ((256, 256), 48, 3),   # 6144, but two lags
    ((128, 128), 64, 7),   # 6144, but no wider than 128
    ((252, 250), 20, 6),   # 6400: swept, lanes and rows past the edge
]


@pytest.mark.parametrize("bc", ["periodic", "neumann"])
@pytest.mark.parametrize("n,m,nh", CASES)
def test_few_lags_match_oracle(n, m, nh, bc):
    from oracle import pyoracle
    p = 1.5
    print("case structure few lags", n, m, nh, bc, flush=True)
    br = BatchRunner("euler2", "none", "hll3", "rungekutta3", bc, [(n + (1,), m)], 1.0, cfl=0.4)
    qs = [smooth_state("euler2", n, seed=70 + s, jump=True) for s in range(3)]
    for s in range(m):
        br.set_state(0, s, qs[s % 3])
    got = br.structure_cube(0, 0, nh, p)
    bound = n[0] * n[1] * 8 * (nh - 1) * 2.0 ** -53
    for s in range(3):
        ref = pyoracle.structure_cube(qs[s][0, 0], bc, nh, p)
        for k in range(s, m, 3):
            assert got[k, 0] == 0
            np.testing.assert_allclose(got[k, 1:], ref[1:], rtol=bound)
