"""The structure function's sweeps and the kinetic energy's split sums at the
sizes where they can go wrong: columns and rows that do not fill a block, lags
too short for a full sweep and lags beyond the domain, every power form, both
boundaries, one sample and several.  All terms are non-negative, so the
relative error of a sum of up to 2e6 of them is below 2e6 * 2^-53 = 2.3e-10
in any order (the oracle sums one after the other)."""
import numpy as np
import pytest

from alsvinn_amd import BatchRunner
from tests.cases import smooth_state

pytestmark = pytest.mark.gpu

CASES = [
    # n, samples, number_of_h, boundary, p
    ((33, 7), 2, 40, "periodic", 2.0),
    ((67, 37), 3, 12, "periodic", 1.0),
    ((64, 32), 1, 34, "neumann", 2.0),
    ((70, 65), 2, 9, "neumann", 3.0),
    ((5, 130), 1, 6, "periodic", 2.5),
    ((129, 3), 2, 5, "neumann", 4.0),
    ((40, 41), 1, 3, "periodic", 5.0),
]


@pytest.mark.parametrize("n,m,nh,bc,p", CASES)
def test_structure_and_energy_match_oracle(n, m, nh, bc, p):
    from oracle import pyoracle
    print("case structure", n, m, nh, bc, p, flush=True)
    br = BatchRunner("euler2", "weno2", "hll3", "rungekutta3", bc, [(n + (1,), m)], 1.0, cfl=0.4)
    qs = [smooth_state("euler2", n, seed=60 + s, jump=True) for s in range(m)]
    for s in range(m):
        br.set_state(0, s, qs[s])
    got = br.structure_cube(0, 0, nh, p)
    ke = br.kinetic_energy(0, 1)
    again = br.structure_cube(0, 0, nh, p)
    np.testing.assert_array_equal(got, again)
    for s in range(m):
        ref = pyoracle.structure_cube(qs[s][0, 0], bc, nh, p)
        assert got[s, 0] == 0
        np.testing.assert_allclose(got[s, 1:], ref[1:], rtol=2.3e-10)
        assert ke[s] == pytest.approx(pyoracle.kinetic_energy(qs[s], 1, 1.0 / (n[0] * n[1])), rel=1e-12)
