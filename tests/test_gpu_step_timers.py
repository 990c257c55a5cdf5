"""avh_time_step_kernels reports the launches that a run of the same solver
makes: one for the whole steps of a small 1D grid, the stage launches where a
tile shape is fixed or the grid is larger; and it advances the solver by the
steps it times."""
import ctypes

import numpy as np
import pytest

import alsvinn_amd
from alsvinn_amd import Simulator, _abi
from tests.cases import smooth_state

pytestmark = pytest.mark.gpu


def _time(s, steps):
    ms = (ctypes.c_double * 4)()
    n = ctypes.c_int()
    _abi.check(alsvinn_amd.load().avh_time_step_kernels(s._h, steps, ms, ctypes.byref(n)))
    return [ms[k] for k in range(n.value)]


@pytest.mark.parametrize("equation,flux,n,integrator,shape,launches", [
    ("burgers", "godunov", 200, "rungekutta3", -1, 1),
    ("burgers", "godunov", 2048, "rungekutta2", -1, 1),
    ("euler1", "hll3", 64, "forwardeuler", -1, 1),
    ("euler1", "hll3", 64, "forwardeuler", 0, 3),
    ("euler1", "hll3", 500, "rungekutta3", 0, 2),
    ("euler1", "hll3", 500, "rungekutta3", 1, 3),
    ("euler1", "hll3", 1200, "rungekutta2", -1, 2),
])
def test_kernels_of_a_step(equation, flux, n, integrator, shape, launches):
    print("case timers", equation, n, integrator, shape, flush=True)

    def solver():
        s = Simulator(equation, "weno2", flux, integrator, "periodic", (n, 1, 1), cfl=0.4)
        s.set_tile_shape(shape)
        s.set_interior(smooth_state(equation, (n,), seed=6))
        return s

    a, b = solver(), solver()
    ms = _time(a, 25)
    assert len(ms) == launches and all(t > 0 for t in ms)
    b.run(max_steps=25)
    assert a.progress().steps == b.progress().steps == 25
    np.testing.assert_array_equal(a.get_interior(), b.get_interior())
