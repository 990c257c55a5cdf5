"""Steps launched past a run's end change nothing: a run whose last chunk is
mostly past its end, and steps enqueued on a solver that has ended, for every
integrator and the launches that test for the end behind their addresses or, past 4096 tiles,
ahead of them."""
import numpy as np
import pytest

from alsvinn_amd import Simulator
from tests.cases import smooth_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("equation,n,flux,shape", [("euler2", (40, 33), "hll3", -1), ("euler2", (40, 33), "hll", 2),
                                                   ("euler2", (70, 45), "hll3", 3), ("euler2", (70, 45), "hll", 4),
                                                   ("euler2", (2050, 955), "hll", 3), ("euler2", (300, 260), "hll", 1),
                                                   ("burgers", (500,), "godunov", 0), ("euler1", (500,), "hll3", 0)])
@pytest.mark.parametrize("integrator", ["forwardeuler", "rungekutta2", "rungekutta3"])
def test_steps_past_the_end(equation, n, flux, shape, integrator):
    print("case idle", equation, n, shape, integrator, flush=True)

    def solver():
        s = Simulator(equation, "weno2", flux, integrator, "periodic", n, cfl=0.3)
        s.set_tile_shape(shape)
        s.set_interior(smooth_state(equation, n, seed=11, jump=False))
        return s

    want, got = solver(), solver()
    for _ in range(3):
        dt = want.perform_step()
    bits = want.get_interior().view(np.uint64)
    end = want.get_current_time()
    p = got.run(end - 0.25 * dt, chunk=64)
    assert (p.steps, p.time) == (3, end)
    for _ in range(2):
        np.testing.assert_array_equal(got.get_interior().view(np.uint64), bits)
        got.enqueue_steps(40)
    # a run with nothing to do, and one more step after it
    p = got.run(end, chunk=64)
    assert (p.steps, p.time) == (3, end)
    want.perform_step()
    p = got.run(1e9, max_steps=1)
    assert p.steps == 4
    np.testing.assert_array_equal(got.get_interior().view(np.uint64), want.get_interior().view(np.uint64))
