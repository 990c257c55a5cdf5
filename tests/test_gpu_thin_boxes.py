"""avh_numerical_flux over boxes of a 3D volume that are a few cells wide:
strips, pencils and corners, on both sides of the line up to which a workgroup
takes one plane (at most one workgroup per compute unit: 64x64 cells are 20
columns, 12 planes of them 240 workgroups), against the oracle bit for bit."""
import ctypes

import numpy as np
import pytest

import alsvinn_amd
from alsvinn_amd import _abi
from alsvinn_amd.simulator import default_context
from tests.devmem import DeviceVolume
from tests.test_gpu_volume import GHOSTS, _cfg, _ivec, _volume_state

pytestmark = pytest.mark.gpu

N = (64, 64, 16)
# start and extent of a box
BOXES = [((0, 0, 0), (2, 2, 2)), ((61, 60, 13), (3, 4, 3)), ((5, 9, 3), (1, 1, 1)), ((0, 31, 7), (64, 2, 2)),
         ((31, 0, 7), (2, 64, 1)), ((17, 15, 0), (2, 2, 16)), ((0, 0, 0), (1, 64, 16)), ((0, 63, 0), (64, 1, 16)),
         ((0, 0, 14), (64, 64, 2)), ((0, 0, 2), (64, 64, 12)), ((0, 0, 2), (64, 64, 13))]


@pytest.mark.parametrize("equation,recon,flux", [("euler3", "weno2", "hll3"), ("euler3", "eno3", "hll"),
                                                 ("euler3", "none", "hll3"), ("euler3", "eno2", "hll3"),
                                                 ("burgers", "weno2", "godunov")])
def test_thin_boxes_bitwise(oracle, equation, recon, flux):
    g = GHOSTS[recon]
    ghosts = (g, g, g)
    cfg, ocfg = _cfg(oracle, equation, recon, flux, N)
    U = _volume_state(equation, tuple(m + 2 * g for m in N), seed=17 + g)
    out0 = np.full_like(U, 44.0)
    dU = DeviceVolume(U, N, ghosts)
    L = alsvinn_amd.load()
    for at, ext in BOXES:
        print("case thin box", equation, recon, at, ext, flush=True)
        end = tuple(at[d] + ext[d] - N[d] for d in range(3))
        dOut = DeviceVolume(out0, N, ghosts)
        ws = (ctypes.c_double * 3)()
        _abi.check(L.avh_numerical_flux(default_context()._h, ctypes.byref(cfg), ctypes.byref(dU.desc),
                                        ctypes.byref(dOut.desc), _ivec(at), _ivec(end), ws, None))
        want, wsw = oracle.compute_flux_box(ocfg, U, out0, at, end)
        np.testing.assert_array_equal(dOut.download(), want)
        np.testing.assert_array_equal(np.array(ws[:]), wsw)
