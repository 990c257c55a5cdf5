"""Parameters and gradients of a network in the caller's order, on both sides of
the size from which parameters are packed on the device (2^17 values with padding):
what set_params wrote comes back from get_params bit for bit, member by member,
and gradients() puts each block where get_params does."""
import numpy as np
import pytest

from alsvinn_amd.surrogate import EnsembleMLP

pytestmark = pytest.mark.gpu

SHAPES = [
    # n_in, n_out, width, hidden, members, batch: values of a member with padding
    (1, 1, 16, 1, 3, 16),      # 544
    (40, 66, 176, 4, 2, 32),   # 116e3
    (40, 66, 192, 4, 2, 32),   # 136e3
    (513, 3, 32, 2, 2, 16),    # layer by layer
]


@pytest.mark.parametrize("shape", SHAPES)
def test_params_and_gradients_in_order(shape):
    from oracle import mlp_oracle as mo
    n_in, n_out, width, hidden, members, batch = shape
    print("case mlp params", shape, flush=True)
    net = EnsembleMLP(n_in, n_out, width=width, hidden=hidden, members=members, batch=batch, seed=2)
    rng = np.random.default_rng(width)
    flats = []
    for m in range(members):
        o = mo.MlpOracle(n_in, width, hidden, n_out)
        o.random_init(rng)
        flats.append(o.flat().astype(np.float32))
        net.set_params(m, flats[m])
    for m in range(members):
        np.testing.assert_array_equal(net.get_params(m), flats[m])
    X = rng.random((batch, n_in)).astype(np.float32)
    Y = rng.normal(size=(batch, n_out)).astype(np.float32)
    net.fit_normalization(X, Y)
    norm = tuple(np.asarray(v, np.float32).astype(np.float64) for v in net.norm)
    _, g = net.gradients(X, Y)
    for m in range(members):
        o.set_flat(flats[m].astype(np.float64))
        _, want, _ = o.loss_and_grads(X, Y, norm, exact=False)
        at = 0
        for r, c in o.shapes:
            for size in (r * c, r):
                # as test_gpu_mlp_fused.py: bf16 products, 2 % a block
                sl = slice(at, at + size)
                assert np.linalg.norm(g[m][sl] - want[sl]) <= 2e-2 * np.linalg.norm(want[sl]) + 1e-7
                at += size
