"""The fused training step and prediction at the shapes where their tiling can
go wrong: layers of one tile and of more tiles than a workgroup has waves, K
with and without a last half step, minibatches of one tile and of several,
row counts that do not fill a tile, one member and several; and the widest
network of the fused path against one just past it (the layer-by-layer path),
which form the same products in the same order.

Tolerances as in test_gpu_mlp.py: gradients against the network oracle in its
bf16-storage mode to 1 % in norm (2 % per block), losses to 1e-3."""
import numpy as np
import pytest

from alsvinn_amd.surrogate import EnsembleMLP

pytestmark = pytest.mark.gpu

SHAPES = [
    # n_in, n_out, width, hidden, members, batch
    (1, 1, 16, 1, 1, 16),
    (40, 66, 256, 4, 2, 48),
    (17, 130, 48, 2, 3, 32),
    (300, 5, 80, 3, 1, 112),
    (33, 290, 272, 2, 2, 16),
    (20, 12, 512, 1, 1, 64),
]


def _net(shape, seed):
    from oracle import mlp_oracle as mo
    n_in, n_out, width, hidden, members, batch = shape
    rng = np.random.default_rng(seed)
    net = EnsembleMLP(n_in, n_out, width=width, hidden=hidden, members=members, batch=batch, seed=seed)
    oracles = []
    for m in range(members):
        o = mo.MlpOracle(n_in, width, hidden, n_out)
        o.random_init(rng)
        o.set_flat(o.flat().astype(np.float32).astype(np.float64))
        net.set_params(m, o.flat())
        oracles.append(o)
    X = rng.random((batch, n_in)).astype(np.float32)
    Y = (rng.normal(size=(batch, n_out)) * 3 + 2).astype(np.float32)
    net.fit_normalization(X, Y)
    norm = tuple(np.asarray(v, np.float32).astype(np.float64) for v in net.norm)
    return net, oracles, X, Y, norm


@pytest.mark.parametrize("shape", SHAPES)
def test_gradients_and_predictions(shape):
    n_in, n_out, width, hidden, members, batch = shape
    print("case fused mlp", shape, flush=True)
    net, oracles, X, Y, norm = _net(shape, 5 + width)
    loss, g = net.gradients(X, Y)
    Xq = np.random.default_rng(1).random((2 * batch + 3, n_in)).astype(np.float32)
    pred = net.predict_members(Xq)
    for m in range(members):
        np.testing.assert_array_equal(net.get_params(m), oracles[m].flat().astype(np.float32))
        lo, go, _ = oracles[m].loss_and_grads(X, Y, norm, exact=False)
        assert loss[m] == pytest.approx(lo, rel=1e-3)
        o = 0
        for (r, c) in oracles[m].shapes:
            for size in (r * c, r):
                sl = slice(o, o + size)
                assert np.linalg.norm(g[m][sl] - go[sl]) <= 2e-2 * np.linalg.norm(go[sl]) + 1e-7
                o += size
        ref = oracles[m].predict(Xq, norm, exact=False)
        assert np.linalg.norm(pred[m] - ref) <= 1e-2 * np.linalg.norm(ref - ref.mean(0)) + 1e-5


def test_training_matches_layerwise_steps():
    """Two epochs of the fused path against the same minibatches through
    gradients() and adam_step() (the update as its own launch)."""
    shape = (40, 66, 256, 2, 1, 16)
    net, _, X, Y, _ = _net(shape, 9)
    other, _, _, _, _ = _net(shape, 9)
    other.set_normalization(*[np.asarray(v, np.float32) for v in net.norm])
    for _ in range(3):  # one minibatch: every order of its rows has the same gradient sums but for rounding
        net.train(X, Y, epochs=1, lr=1e-3, final_lr_fraction=1.0)
        other.gradients(X, Y)
        other.adam_step(1e-3)
    a, b = net.get_params(0), other.get_params(0)
    # Adam moves a parameter by at most lr a step, and rounding can flip the
    # direction of one whose gradient is zero to rounding
    assert np.abs(a - b).max() <= 3 * 2 * 1e-3
    assert np.linalg.norm(a - b) <= 1e-3 * np.linalg.norm(a)


def test_row_counts_of_predictions():
    shape = (40, 66, 64, 2, 3, 64)
    net, _, _, _, _ = _net(shape, 3)
    X = np.random.default_rng(2).random((200, 40)).astype(np.float32)
    whole = net.predict_members(X)
    for rows in (1, 15, 16, 17, 199):
        np.testing.assert_array_equal(net.predict_members(X[:rows]), whole[:, :rows])
