"""RK3's last two stages in one launch (shape 2 of 2D grids, shape 0 of 1D
ones): the oracle's bits on ragged tiles, at the shortest axes the launch takes
and just below them, where the separate stages run, with both boundaries; a
violation stops at the same step with the same state."""
import numpy as np
import pytest

import alsvinn_amd
from tests.cases import smooth_state

pytestmark = pytest.mark.gpu

SIZES = {1: [(5,), (6,), (240,), (241,), (1500,)],
         2: [(5, 40), (6, 6), (40, 5), (16, 7), (17, 15), (33, 31), (66, 47)]}


@pytest.mark.parametrize("recon", ["none", "weno2", "eno2", "eno3"])
@pytest.mark.parametrize("equation,flux", [("burgers", "godunov"), ("euler1", "hll3"), ("euler2", "hll3"),
                                           ("euler2", "hll"), ("euler3", "hll3")])
def test_last_two_stages_bitwise(equation, flux, recon):
    from oracle import pyoracle
    dims = (1, 2) if equation == "burgers" else ((1,) if equation == "euler1" else (2,))
    for dim in dims:
        for n in SIZES[dim]:
            for bc in ("periodic", "neumann"):
                full = n + (1,) * (3 - dim)
                q0 = smooth_state(equation, n, seed=sum(n), jump=True)
                o = pyoracle.Simulator(equation, recon, flux, "rungekutta3", bc, full, cfl=0.35)
                o.set_interior(q0)
                for _ in range(5):
                    o.step()
                for shape in (2,) if dim == 2 else (0,):
                    print("case pair", equation, flux, recon, n, bc, shape, flush=True)
                    h = alsvinn_amd.Simulator(equation, recon, flux, "rungekutta3", bc, full, cfl=0.35)
                    h.set_tile_shape(shape)
                    h.set_interior(q0)
                    for _ in range(5):
                        h.perform_step()
                    np.testing.assert_array_equal(h.get_interior().view(np.uint64), o.get_interior().view(np.uint64))
                    assert h.progress().time == o.time


def test_violation_stops_as_separate_stages_do():
    runs = []
    for shape in (2, 3):
        h = alsvinn_amd.Simulator("euler2", "weno2", "hll", "rungekutta3", "periodic", (50, 41), cfl=2.5)
        h.set_tile_shape(shape)
        h.set_interior(smooth_state("euler2", (50, 41), seed=5, jump=True))
        h.enqueue_steps(60)
        runs.append((h.get_interior(), h.progress()))
    (got, q), (want, p) = runs
    assert p.violated == 1
    assert (q.steps, q.violated, q.time) == (p.steps, p.violated, p.time)
    nan = np.isnan(want)
    np.testing.assert_array_equal(np.isnan(got), nan)
    np.testing.assert_array_equal(got[~nan].view(np.uint64), want[~nan].view(np.uint64))
