"""Device memory of a network: one that trains by the fused launches holds what
these use (weights and moments, gelu' and transposed activations of every hidden
layer, transposed dZ of every layer) and not the buffers of the layer-by-layer
path beside them."""
import ctypes

import pytest

from alsvinn_amd.surrogate import EnsembleMLP
from tests.devmem import hip

pytestmark = pytest.mark.gpu


def _free():
    f, t = ctypes.c_size_t(), ctypes.c_size_t()
    hip().hipDeviceSynchronize()
    assert hip().hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
    return f.value


def test_fused_network_holds_what_it_uses():
    n_in, n_out, width, hidden, members, batch = 40, 66, 512, 7, 8, 4096
    EnsembleMLP(1, 1, width=16, hidden=1, members=1, batch=16)  # the library's own first allocations
    before = _free()
    net = EnsembleMLP(n_in, n_out, width=width, hidden=hidden, members=members, batch=batch)
    used = before - _free()
    weights = 48 * width + (hidden - 1) * width * width + width * 80
    params = weights + hidden * width + 80
    need = members * (4 * 4 * params + 2 * 2 * weights)               # p, m, v, gradients; bf16 weights twice
    need += members * batch * (hidden * width * (4 + 2) + 48 * 2)     # gelu', transposed activations, inputs
    need += members * batch * (hidden + 1) * width * 2                # transposed dZ
    print("case mlp memory", used, need, flush=True)
    assert used <= need + (64 << 20)  # a few small arrays, and each allocation rounded up to 2 MiB
    del net
