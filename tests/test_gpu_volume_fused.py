"""Substeps whose dt is given combine in the stage kernel's write-back; the
net flux from avh_numerical_flux and the integrator's Volume operations in
numpy must give the same bits on every cell, ghost cells included: several
tiles and chunks, ragged edges, more ghost cells than the stencil needs, and an
output that shares memory with an input (which keeps the separate passes)."""
import ctypes

import numpy as np
import pytest

import alsvinn_amd
from alsvinn_amd import _abi
from alsvinn_amd.simulator import default_context
from tests.devmem import DeviceVolume
from tests.test_gpu_volume import GHOSTS, _cfg, _ivec, _volume_state

pytestmark = pytest.mark.gpu

CASES = [("burgers", "weno2", "godunov", (300, 1, 1)), ("euler1", "eno3", "hll", (257, 1, 1)),
         ("burgers", "none", "godunov", (35, 17, 1)), ("euler2", "weno2", "hll3", (65, 47, 1)),
         ("burgers", "eno2", "godunov", (17, 16, 5)), ("euler3", "none", "hll", (16, 15, 3)),
         ("euler3", "weno2", "hll3", (33, 31, 70)), ("euler3", "eno3", "hll3", (17, 46, 21)),
         ("euler3", "weno2", "hll3", (27, 33, 40)), ("euler3", "eno2", "hll", (32, 28, 19))]


def _combine(integ, substep, L, us, u0, s):
    o = L * s + us
    if integ == "rungekutta2":
        return (o + u0) * 0.5
    if substep == 1:
        return (o * (1.0 / 3.0) + u0) * (3.0 / 4.0)
    return (o * 2 + u0) * (1.0 / 3.0)


@pytest.mark.parametrize("extra", [0, 2])
@pytest.mark.parametrize("equation,recon,flux,n", CASES)
def test_fused_substeps_bitwise(oracle, equation, recon, flux, n, extra):
    dim = 3 if n[2] > 1 else (2 if n[1] > 1 else 1)
    ghosts = tuple(GHOSTS[recon] + extra if d < dim else 0 for d in range(3))
    if any(n[d] < ghosts[d] for d in range(dim)):
        ghosts = tuple(GHOSTS[recon] if d < dim else 0 for d in range(3))
    total = tuple(n[d] + 2 * ghosts[d] for d in range(3))
    L, ctx = alsvinn_amd.load(), default_context()
    u = [_volume_state(equation, total, seed=k) for k in range(3)]
    at = (slice(None),) + tuple(slice(ghosts[d], total[d] - ghosts[d]) for d in (2, 1, 0))
    dt = 1e-3
    for integ, substep in (("rungekutta2", 1), ("rungekutta3", 1), ("rungekutta3", 2)):
        cfg, _ = _cfg(oracle, equation, recon, flux, n, integ=integ)
        s = dt / ((cfg.upper[0] - cfg.lower[0]) / n[0])
        old = _volume_state(equation, total, seed=7)
        for alias in (False, True):
            print("case fused", equation, recon, flux, n, ghosts, integ, substep, alias, flush=True)
            vols = [DeviceVolume(x, n, ghosts) for x in u]
            out = vols[0] if alias else DeviceVolume(old, n, ghosts)
            flux_out = DeviceVolume(u[0] if alias else old, n, ghosts)
            ws = (ctypes.c_double * 3)()
            _abi.check(L.avh_numerical_flux(ctx._h, ctypes.byref(cfg), ctypes.byref(vols[substep].desc),
                                            ctypes.byref(flux_out.desc), _ivec((0, 0, 0)), _ivec((0, 0, 0)), ws,
                                            None))
            net = flux_out.download()
            u0 = u[0]
            if alias:  # the combination then finds the net flux in U0's place
                u0 = u0.copy()
                u0[at] = net[at]
            want = _combine(integ, substep, net, u[substep], u0, s)
            inputs = (ctypes.POINTER(_abi.AvhVolume) * (substep + 1))(
                *[ctypes.pointer(v.desc) for v in vols[:substep + 1]])
            got_dt = ctypes.c_double(0.0)
            _abi.check(L.avh_substep(ctx._h, ctypes.byref(cfg), inputs, substep, ctypes.byref(out.desc), dt,
                                     float("inf"), ctypes.byref(got_dt), None))
            assert got_dt.value == dt
            np.testing.assert_array_equal(out.download().view(np.uint64), want.view(np.uint64))
