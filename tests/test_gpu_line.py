"""Small 1D grids run their steps in one workgroup; a fixed tile shape asks
for the stage kernels.  Both must give the same bits -- states, times, step
counts, save counters -- over every scheme, at the edges of the thread and
wavefront counts and of the sizes the rule admits, with saves that clip dt,
pauses, a constraint violation in the middle, and state that is not finite."""
import numpy as np
import pytest

import alsvinn_amd
from tests.cases import NV, smooth_state

pytestmark = pytest.mark.gpu

SCHEMES = [("burgers", "godunov")] + [("euler1", f) for f in ("hll", "hll3")]
SIZES = [3, 62, 63, 64, 65, 200, 1022, 1023, 1024, 1025, 2047, 2048, 2049]


def _pair(eq, recon, flux, integ, bc, n, cfl=0.4):
    pair = [alsvinn_amd.Simulator(eq, recon, flux, integ, bc, (n,), cfl=cfl) for _ in range(2)]
    pair[1].set_tile_shape(0)
    return pair


def _same_bits(a, b):
    """The same bits, NaN where the other has NaN: IEEE 754 leaves the sign
    and payload of a NaN result open."""
    nan = np.isnan(b)
    np.testing.assert_array_equal(np.isnan(a), nan)
    np.testing.assert_array_equal(a[~nan].view(np.uint64), b[~nan].view(np.uint64))


def _same(a, b):
    _same_bits(a.get_state(), b.get_state())
    p, q = a.progress(), b.progress()
    assert (p.steps, p.violated, p.saves_pending) == (q.steps, q.violated, q.saves_pending)
    assert np.float64(p.time).view(np.uint64) == np.float64(q.time).view(np.uint64)
    assert np.float64(p.last_dt).view(np.uint64) == np.float64(q.last_dt).view(np.uint64)


@pytest.mark.parametrize("recon", ["none", "weno2", "eno2", "eno3"])
@pytest.mark.parametrize("scheme", SCHEMES, ids=lambda s: s[0] + "-" + s[1])
def test_steps_in_one_workgroup_bitwise(scheme, recon):
    eq, flux = scheme
    for integ in ("forwardeuler", "rungekutta2", "rungekutta3"):
        for bc in ("periodic", "neumann"):
            for n in SIZES:
                print("case", eq, flux, recon, integ, bc, n, flush=True)
                pair = _pair(eq, recon, flux, integ, bc, n)
                for s in pair:
                    s.set_interior(smooth_state(eq, (n,), seed=n, jump=True))
                    s.perform_step()
                    s.enqueue_steps(21)
                _same(*pair)


def test_saves_pauses_and_end():
    """Two writers; the run pauses at every save, lands on the end time and a
    second run goes on from there."""
    for n in (200, 1024):
        pair = _pair("euler1", "weno2", "hll3", "rungekutta3", "neumann", n)
        for s in pair:
            s.add_fixed_interval_writer(0.004)
            s.add_fixed_interval_writer(0.007, 0.001, True)
            s.set_interior(smooth_state("euler1", (n,), seed=2, jump=True))
        for _ in range(6):
            for s in pair:
                s.run(0.05, chunk=13, pause_on_save=True)
            _same(*pair)
            for s in pair:
                s.ack_saves()
        for t in (0.05, 0.06):
            for s in pair:
                s.run(t, max_steps=5000, chunk=13)
            _same(*pair)


@pytest.mark.parametrize("integ", ["forwardeuler", "rungekutta2", "rungekutta3"])
def test_violation_stops_both(integ):
    """Too long a step breaks positivity after some steps."""
    pair = _pair("euler1", "eno2", "hll", integ, "periodic", 130, cfl=2.5)
    for s in pair:
        s.set_interior(smooth_state("euler1", (130,), seed=5, jump=True))
        s.enqueue_steps(200)
    assert pair[1].progress().violated == 1
    _same(*pair)


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf, 1e-320, -0.0])
def test_unusual_values(value):
    for eq, flux in SCHEMES:
        pair = _pair(eq, "weno2", flux, "rungekutta3", "periodic", 100)
        for s in pair:
            q = smooth_state(eq, (100,), seed=1, jump=True)
            q[NV[eq] - 1].reshape(-1)[37:40] = value
            s.set_interior(q)
            s.enqueue_steps(3)
        _same_bits(*(s.get_state() for s in pair))
        p, q = (s.progress() for s in pair)
        assert (p.steps, p.violated) == (q.steps, q.violated)
