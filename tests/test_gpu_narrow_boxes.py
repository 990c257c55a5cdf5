"""Boxes of a 3D volume at most four cells wide in x, which have columns of
their own (4x24 cells, as many planes a workgroup as leave 1024 workgroups), and
ones of five, which have not: avh_numerical_flux against the oracle bit for bit,
and substeps of grids that narrow."""
import ctypes

import numpy as np
import pytest

import alsvinn_amd
import tests.test_gpu_volume_fused as fused
from alsvinn_amd import _abi
from alsvinn_amd.simulator import default_context
from tests.devmem import DeviceVolume
from tests.test_gpu_volume import GHOSTS, _cfg, _ivec, _volume_state

pytestmark = pytest.mark.gpu

N = (6, 50, 400)
# start and extent of a box: 3 columns of 400 planes go two planes a workgroup
BOXES = [((0, 0, 0), (2, 50, 400)), ((3, 0, 3), (3, 49, 397)), ((2, 1, 0), (4, 25, 33)), ((5, 26, 1), (1, 24, 1)),
         ((0, 0, 399), (4, 48, 1)), ((1, 7, 5), (2, 1, 200)), ((0, 30, 17), (1, 2, 3)), ((1, 0, 0), (5, 25, 30))]
CASES = [("euler3", "weno2", "hll3"), ("euler3", "eno3", "hll"), ("euler3", "none", "hll3"), ("euler3", "eno2", "hll"),
         ("burgers", "weno2", "godunov")]


@pytest.mark.parametrize("equation,recon,flux", CASES)
def test_narrow_boxes_bitwise(oracle, equation, recon, flux):
    g = GHOSTS[recon]
    ghosts = (g, g, g)
    cfg, ocfg = _cfg(oracle, equation, recon, flux, N)
    U = _volume_state(equation, tuple(m + 2 * g for m in N), seed=23 + g)
    out0 = np.full_like(U, 44.0)
    dU = DeviceVolume(U, N, ghosts)
    L = alsvinn_amd.load()
    for at, ext in BOXES:
        print("case narrow box", equation, recon, at, ext, flush=True)
        end = tuple(at[d] + ext[d] - N[d] for d in range(3))
        dOut = DeviceVolume(out0, N, ghosts)
        ws = (ctypes.c_double * 3)()
        _abi.check(L.avh_numerical_flux(default_context()._h, ctypes.byref(cfg), ctypes.byref(dU.desc),
                                        ctypes.byref(dOut.desc), _ivec(at), _ivec(end), ws, None))
        want, wsw = oracle.compute_flux_box(ocfg, U, out0, at, end)
        np.testing.assert_array_equal(dOut.download(), want)
        np.testing.assert_array_equal(np.array(ws[:]), wsw)


@pytest.mark.parametrize("equation,recon,flux,n", [("euler3", "weno2", "hll3", (4, 25, 11)),
                                                   ("euler3", "eno3", "hll", (3, 49, 7)),
                                                   ("euler3", "none", "hll3", (2, 24, 600)),
                                                   ("burgers", "eno2", "godunov", (4, 23, 9))])
def test_narrow_substeps_bitwise(oracle, equation, recon, flux, n):
    fused.test_fused_substeps_bitwise(oracle, equation, recon, flux, n, 0)
