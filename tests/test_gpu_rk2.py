"""RK2's second stage forms U1 while it loads, from L0 and a copy of U0 that
the first stage writes: every tile shape against the oracle bit for bit, on
grids with ragged edges and several tiles (2D) and chunks (3D), and batches on
every shape against single runs."""
import numpy as np
import pytest

import alsvinn_amd
from alsvinn_amd.uq import BatchRunner
from tests.cases import smooth_state

pytestmark = pytest.mark.gpu

CASES = [("euler2", "weno2", "hll3", "periodic", (67, 49)), ("euler2", "eno3", "hll", "neumann", (33, 31)),
         ("burgers", "none", "godunov", "neumann", (40, 18)), ("euler3", "weno2", "hll3", "neumann", (35, 17, 11)),
         ("euler3", "eno2", "hll", "periodic", (18, 31, 9)), ("euler1", "weno2", "hll3", "periodic", (1500,))]


@pytest.mark.parametrize("equation,recon,flux,bc,n", CASES)
def test_rk2_every_shape_bitwise(equation, recon, flux, bc, n):
    from oracle import pyoracle
    q0 = smooth_state(equation, n, seed=21, jump=True)
    full = tuple(n) + (1,) * (3 - len(n))
    o = pyoracle.Simulator(equation, recon, flux, "rungekutta2", bc, full, cfl=0.35)
    o.set_interior(q0)
    for _ in range(7):
        o.step()
    for shape in range((2, 5, 7)[len(n) - 1]):
        print("case rk2", equation, recon, flux, bc, n, shape, flush=True)
        h = alsvinn_amd.Simulator(equation, recon, flux, "rungekutta2", bc, full, cfl=0.35)
        h.set_tile_shape(shape)
        h.set_interior(q0)
        for _ in range(7):
            h.perform_step()
        np.testing.assert_array_equal(h.get_interior().view(np.uint64), o.get_interior().view(np.uint64))
        assert h.progress().time == o.time


@pytest.mark.parametrize("n", [(45, 34), (300,)])
def test_rk2_batches_match_single_runs(n):
    full = tuple(n) + (1,) * (3 - len(n))
    equation = "euler%d" % len(n)
    states = [smooth_state(equation, n, seed=s, jump=True) for s in range(3)]
    want = []
    for q in states:
        h = alsvinn_amd.Simulator(equation, "weno2", "hll3", "rungekutta2", "periodic", full, cfl=0.4)
        h.set_interior(q)
        h.enqueue_steps(9)
        want.append(h.get_interior())
    for shape in range((2, 5)[len(n) - 1]):
        print("case rk2 batch", n, shape, flush=True)
        br = BatchRunner(equation, "weno2", "hll3", "rungekutta2", "periodic", [(n, 3)], 1e9, cfl=0.4, stats_saves=0)
        br.set_tile_shape(shape)
        for s, q in enumerate(states):
            br.set_state(0, s, q)
        assert br.run(max_steps=9, chunk=9)[0] == 9
        for s in range(3):
            np.testing.assert_array_equal(br.get_state(0, s).reshape(want[s].shape).view(np.uint64),
                                          want[s].view(np.uint64))
