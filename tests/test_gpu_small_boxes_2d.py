"""2D boxes on both sides of the line up to which they take 16x7 tiles instead
of 32x15 ones (384 of the former): whole volumes, strips, pencils of one cell
and ragged edges, against the oracle bit for bit."""
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

N = (257, 175, 1)
# start and extent of a box; 16x7 tiles: 16 x 24 are 384, one more row 400
BOXES = [((0, 0), (256, 168)), ((1, 2), (256, 169)), ((0, 0), (257, 175)), ((0, 0), (2, 175)), ((254, 0), (3, 175)),
         ((0, 173), (257, 2)), ((100, 50), (1, 1)), ((3, 5), (17, 8)), ((0, 0), (16, 7)), ((240, 160), (15, 15))]
CASES = [("euler2", "weno2", "hll3"), ("euler2", "eno3", "hll"), ("euler3", "none", "hll3"), ("euler2", "eno2", "hll"),
         ("burgers", "weno2", "godunov")]


@pytest.mark.parametrize("equation,recon,flux", CASES)
def test_boxes_bitwise(oracle, equation, recon, flux):
    g = GHOSTS[recon]
    ghosts = (g, g, 0)
    cfg, ocfg = _cfg(oracle, equation, recon, flux, N)
    U = _volume_state(equation, (N[0] + 2 * g, N[1] + 2 * g, 1), seed=31 + g)
    out0 = np.full_like(U, 44.0)
    dU = DeviceVolume(U, N, ghosts)
    L = alsvinn_amd.load()
    for at, ext in BOXES:
        print("case box", equation, recon, at, ext, flush=True)
        at, end = at + (0,), tuple(at[d] + ext[d] - N[d] for d in range(2)) + (0,)
        dOut = DeviceVolume(out0, N, ghosts)
        ws = (ctypes.c_double * 3)()
        _abi.check(L.avh_numerical_flux(default_context()._h, ctypes.byref(cfg), ctypes.byref(dU.desc),
                                        ctypes.byref(dOut.desc), _ivec(at), _ivec(end), ws, None))
        want, wsw = oracle.compute_flux_box(ocfg, U, out0, at, end)
        np.testing.assert_array_equal(dOut.download(), want)
        np.testing.assert_array_equal(np.array(ws[:]), wsw)


@pytest.mark.parametrize("equation,recon,flux,n", [("euler2", "weno2", "hll3", (256, 168, 1)),
                                                   ("euler2", "eno3", "hll", (256, 169, 1))])
def test_substeps_bitwise(oracle, equation, recon, flux, n):
    fused.test_fused_substeps_bitwise(oracle, equation, recon, flux, n, 0)
