"""Kinetic energy of batches on both sides of the sample size up to which one
block holds a sample and scales its sum itself (2048 cells), against the oracle.
The terms are non-negative: the relative error of a sum of n of them is below
n * 2^-53 in any order, and a few 2^-53 come with the scale."""
import numpy as np
import pytest

from alsvinn_amd import BatchRunner
from tests.cases import smooth_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("equation,n,m", [("euler1", (200,), 100), ("euler1", (1,), 3), ("euler1", (2048,), 2),
                                          ("euler1", (2049,), 2), ("euler2", (64, 32), 5), ("euler2", (64, 33), 5)])
def test_kinetic_energy_matches_oracle(equation, n, m):
    from oracle import pyoracle
    print("case kinetic energy", equation, n, m, flush=True)
    br = BatchRunner(equation, "none", "hll3", "rungekutta3", "periodic", [(n, m)], 1.0, cfl=0.4)
    qs = [smooth_state(equation, n, seed=30 + s, jump=True) for s in range(3)]
    for s in range(m):
        br.set_state(0, s, qs[s % 3])
    cells = int(np.prod(n))
    dv = np.prod([1.0 / k for k in n if k > 1])
    for comp in range(len(n)):
        got = br.kinetic_energy(0, comp)
        for s in range(m):
            want = pyoracle.kinetic_energy(qs[s % 3], comp, dv)
            assert got[s] == pytest.approx(want, rel=(cells + 8) * 2.0 ** -53)
