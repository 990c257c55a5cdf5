"""The 2D structure function on both sides of the lines between its two ways, a
thread a cell and the column sweep: few lags and few pairs of cells, and for a
general power grids that fill the sweep's lanes in enough blocks.  All terms are
non-negative, so the relative error of a sum of n of them is below n * 2^-53 in
any order (the oracle sums one after the other), and a general power adds a few
2^-53 a term."""
import numpy as np
import pytest

from alsvinn_amd import BatchRunner
from tests.cases import smooth_state

pytestmark = pytest.mark.gpu

CASES = [
    # n, samples, number_of_h, p; which side of the line is said behind
    ((31, 45), 2, 13, 2.0),      # 12 lags: a thread a cell
    ((31, 45), 2, 14, 2.0),      # 13: swept
    ((299, 291), 4, 4, 1.0),     # 16.7e6 pairs: just below 2^24
    ((299, 301), 4, 4, 4.0),     # 17.3e6
    ((17, 60), 3, 30, 2.5),      # a general power on a narrow grid
    ((1, 61), 2, 9, 2.5),
    ((128, 128), 15, 9, 1.5),    # 1920 blocks
    ((128, 128), 16, 9, 1.5),    # 2048: swept
    ((129, 128), 16, 9, 2.5),    # lanes past the edge
]


@pytest.mark.parametrize("bc", ["periodic", "neumann"])
@pytest.mark.parametrize("n,m,nh,p", CASES)
def test_structure_routes_match_oracle(n, m, nh, p, bc):
    from oracle import pyoracle
    print("case structure route", n, m, nh, bc, p, flush=True)
    br = BatchRunner("euler2", "none", "hll3", "rungekutta3", bc, [(n + (1,), m)], 1.0, cfl=0.4)
    qs = [smooth_state("euler2", n, seed=90 + s, jump=True) for s in range(3)]
    for s in range(m):
        br.set_state(0, s, qs[s % 3])
    got = br.structure_cube(0, 0, nh, p)
    np.testing.assert_array_equal(got, br.structure_cube(0, 0, nh, p))
    bound = n[0] * n[1] * 8 * (nh - 1) * 2.0 ** -53
    for s in range(min(m, 3)):
        ref = pyoracle.structure_cube(qs[s][0, 0], bc, nh, p)
        for k in range(s, m, 3):
            assert got[k, 0] == 0
            np.testing.assert_allclose(got[k, 1:], ref[1:], rtol=bound)
