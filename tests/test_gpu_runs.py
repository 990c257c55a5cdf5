"""A run opens on the device: what it does must not depend on what the host saw
last -- steps enqueued without a look in between, an end time already reached,
pending saves, a broken constraint -- on the one-workgroup path, captured steps
and plain launches."""
import numpy as np
import pytest

import alsvinn_amd
from alsvinn_amd import _abi
from tests.cases import smooth_state

pytestmark = pytest.mark.gpu

GRIDS = [("euler1", (150,), "hll3"), ("euler2", (40, 22), "hll3")]


def _sim(equation, n, flux, cfl=0.4):
    s = alsvinn_amd.Simulator(equation, "weno2", flux, "rungekutta3", "periodic", n, cfl=cfl)
    s.set_interior(smooth_state(equation, n, seed=4, jump=True))
    return s


@pytest.mark.parametrize("graph_steps", [0, 4])
@pytest.mark.parametrize("equation,n,flux", GRIDS)
def test_runs_after_unseen_steps(equation, n, flux, graph_steps):
    want, got = _sim(equation, n, flux), _sim(equation, n, flux)
    for _ in range(17):
        want.perform_step()
    got.set_graph_steps(graph_steps)
    print("case runs", equation, n, graph_steps, flush=True)
    got.enqueue_steps(5)
    p = got.run(1e9, max_steps=9, chunk=4)
    assert p.steps == 14
    got.enqueue_steps(3)
    np.testing.assert_array_equal(got.get_interior().view(np.uint64), want.get_interior().view(np.uint64))
    # the end time has passed without the host having seen it
    t = got.progress().time
    got.enqueue_steps(1)
    p = got.run(t, max_steps=5)
    assert p.steps == 18 and p.time > t
    assert got.run(t, max_steps=0).steps == 18
    # and on again to a later one, landing on the run's own count of steps
    p = got.run(1e9, max_steps=6, chunk=6)
    assert p.steps == 24


@pytest.mark.parametrize("equation,n,flux", GRIDS)
def test_pending_saves_hold_a_run(equation, n, flux):
    s = _sim(equation, n, flux)
    s.add_fixed_interval_writer(1e-3)
    p = s.run(1.0, max_steps=500, pause_on_save=True)
    assert p.saves_pending == 1
    q = s.run(1.0, max_steps=500, pause_on_save=True)
    assert (q.steps, q.time) == (p.steps, p.time)
    s.ack_saves()
    q = s.run(1.0, max_steps=500, pause_on_save=True)
    assert q.steps > p.steps and q.saves_pending == 1


@pytest.mark.parametrize("equation,n,flux", GRIDS)
def test_a_broken_run_stays_broken(equation, n, flux):
    s = _sim(equation, n, flux, cfl=3.0)
    s.enqueue_steps(150)
    for _ in range(2):
        with pytest.raises(_abi.ConstraintError):
            s.run(1e9, max_steps=10)
    p = s.progress()
    assert p.violated == 1 and p.steps < 150
