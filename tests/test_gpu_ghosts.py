"""avh_apply_boundary on both sides of the number of ghost cells from which a
thread copies every variable (2^17): flat volumes, whose ghost planes are most of
them, and one to five variables, against the oracle bit for bit."""
import ctypes

import numpy as np
import pytest

import alsvinn_amd
from alsvinn_amd import _abi
from alsvinn_amd.simulator import default_context
from tests.devmem import DeviceVolume
from tests.test_gpu_volume import _cfg

pytestmark = pytest.mark.gpu

CASES = [
    # equation, reconstruction (its ghost cells), cells; ghost cells in all
    ("euler3", "weno2", (175, 175, 2)),   # 130996: one variable a block
    ("euler3", "weno2", (176, 175, 2)),   # 131720: together
    ("euler3", "eno3", (130, 131, 40)),
    ("burgers", "weno2", (181, 175, 3)),
    ("euler2", "weno2", (33000, 2, 1)),
]


@pytest.mark.parametrize("bc", ["periodic", "neumann"])
@pytest.mark.parametrize("equation,recon,n", CASES)
def test_ghost_cells_bitwise(oracle, equation, recon, n, bc):
    g = {"weno2": 2, "eno3": 3}[recon]
    dim = 3 if n[2] > 1 else 2
    ghosts = tuple(g if d < dim else 0 for d in range(3))
    total = tuple(n[d] + 2 * ghosts[d] for d in range(3))
    cells = total[0] * total[1] * total[2] - n[0] * n[1] * n[2]
    print("case ghosts", equation, n, bc, cells, flush=True)
    nv = {"burgers": 1, "euler2": 4, "euler3": 5}[equation]
    flux = "godunov" if equation == "burgers" else "hll3"
    _, ocfg = _cfg(oracle, equation, recon, flux, n, bc=bc)
    U = np.random.default_rng(cells).random((nv, total[2], total[1], total[0]))
    dU = DeviceVolume(U, n, ghosts)
    _abi.check(alsvinn_amd.load().avh_apply_boundary(default_context()._h, {"periodic": 0, "neumann": 1}[bc],
                                                     ctypes.byref(dU.desc), None))
    np.testing.assert_array_equal(dU.download(), oracle.apply_boundary(ocfg, g, U))
