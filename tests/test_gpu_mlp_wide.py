"""Networks past the widest that the fused launches serve (512 inputs, outputs
or neurons a layer), which run layer by layer: loss, gradients, Adam steps,
predictions and training against the network oracle in its bf16-storage mode;
and, for both kinds, the update that training makes against gradients() and
adam_step() on the same rows.

Tolerances: gradients, losses and predictions as in test_gpu_mlp.py (1 % in
norm, 2 % a block, 1e-3), Adam steps 2e-5.  Training visits the rows of its one
minibatch in another order than gradients(), so sums differ by rounding alone;
Adam's first steps are about lr whatever the gradient's size, so a parameter
differs by more than a hundredth of lr only where its gradient is rounding
itself, a share well below one in a hundred."""
import numpy as np
import pytest

from alsvinn_amd.surrogate import EnsembleMLP

pytestmark = pytest.mark.gpu

WIDE = [
    # n_in, n_out, width, hidden, members, batch
    (40, 66, 528, 2, 2, 48),
    (513, 12, 64, 2, 2, 32),
    (20, 513, 48, 1, 3, 16),
    (600, 530, 544, 1, 1, 16),
]


def _net(shape, seed, big_biases=False):
    from oracle import mlp_oracle as mo
    n_in, n_out, width, hidden, members, batch = shape
    rng = np.random.default_rng(seed)
    net = EnsembleMLP(n_in, n_out, width=width, hidden=hidden, members=members, batch=batch, seed=seed)
    oracles = []
    for m in range(members):
        o = mo.MlpOracle(n_in, width, hidden, n_out)
        o.random_init(rng)
        flat = o.flat()
        if big_biases:
            b = ~o.weight_mask().astype(bool)
            flat[b] = rng.normal(size=b.sum())
        o.set_flat(flat.astype(np.float32).astype(np.float64))
        net.set_params(m, o.flat())
        oracles.append(o)
    X = rng.random((batch, n_in)).astype(np.float32)
    Y = (rng.normal(size=(batch, n_out)) * 3 + 2).astype(np.float32)
    net.fit_normalization(X, Y)
    norm = tuple(np.asarray(v, np.float32).astype(np.float64) for v in net.norm)
    return net, oracles, X, Y, norm


@pytest.mark.parametrize("shape", WIDE)
def test_wide_gradients_steps_and_predictions(shape):
    from oracle import mlp_oracle as mo
    n_in, n_out, width, hidden, members, batch = shape
    print("case wide mlp", shape, flush=True)
    net, oracles, X, Y, norm = _net(shape, 3 + width)
    Xq = np.random.default_rng(1).random((2 * batch + 3, n_in)).astype(np.float32)
    pred = net.predict_members(Xq)
    net.set_weight_decay(0.05)
    mask = oracles[0].weight_mask()
    p = [net.get_params(m).astype(np.float64) for m in range(members)]
    mst = [np.zeros_like(x) for x in p]
    vst = [np.zeros_like(x) for x in p]
    for t in (1, 2):
        loss, g = net.gradients(X, Y)
        for m in range(members):
            oracles[m].set_flat(p[m])
            lo, go, _ = oracles[m].loss_and_grads(X, Y, norm, exact=False)
            assert loss[m] == pytest.approx(lo, rel=1e-3)
            assert np.linalg.norm(g[m] - go) <= 1e-2 * np.linalg.norm(go)
            o = 0
            for (r, c) in oracles[m].shapes:
                for size in (r * c, r):
                    sl = slice(o, o + size)
                    assert np.linalg.norm(g[m][sl] - go[sl]) <= 2e-2 * np.linalg.norm(go[sl]) + 1e-7
                    o += size
            if t == 1:
                ref = oracles[m].predict(Xq, norm, exact=False)
                assert np.linalg.norm(pred[m] - ref) <= 1e-2 * np.linalg.norm(ref - ref.mean(0)) + 1e-5
        net.adam_step(1e-3)
        for m in range(members):
            p[m], mst[m], vst[m] = mo.adam(p[m], g[m].astype(np.float64), mst[m], vst[m], t, 1e-3,
                                           weight_decay=0.05, decay_mask=mask)
            got = net.get_params(m).astype(np.float64)
            np.testing.assert_allclose(got, p[m], rtol=2e-5, atol=2e-7)
            p[m] = got


@pytest.mark.parametrize("shape", [(40, 66, 256, 2, 2, 32), (17, 130, 48, 3, 3, 64), (40, 66, 528, 2, 2, 32),
                                   (513, 12, 64, 2, 2, 32)])
def test_training_makes_the_steps_of_gradients_and_adam(shape):
    """Three steps of one minibatch, weight decay 1 and biases of about 1, so
    that a decay on the biases, or one left out of the weights, shows."""
    print("case mlp update", shape, flush=True)
    lr = 1e-3
    net, oracles, X, Y, _ = _net(shape, 9, big_biases=True)
    other, _, _, _, _ = _net(shape, 9, big_biases=True)
    other.set_normalization(*[np.asarray(v, np.float32) for v in net.norm])
    for n in (net, other):
        n.set_weight_decay(1.0)
    for _ in range(3):
        hist = net.train(X, Y, epochs=1, lr=lr, final_lr_fraction=1.0)
        loss, _ = other.gradients(X, Y)
        other.adam_step(lr)
        np.testing.assert_allclose(hist[0], loss, rtol=1e-3)
    weights = oracles[0].weight_mask().astype(bool)
    for m in range(shape[4]):
        start, a, b = oracles[m].flat(), net.get_params(m), other.get_params(m)
        for part in (weights, ~weights):
            off = np.abs(a[part] - b[part])
            assert np.mean(off > 1e-2 * lr) < 1e-2
            # and they moved
            assert np.median(np.abs(a[part] - start[part])) > lr


def test_wide_training_lowers_the_loss():
    rng = np.random.default_rng(4)
    X = rng.random((200, 6)).astype(np.float32)
    Y = np.stack([np.sin(3 * X[:, 0]) + X[:, 1], X[:, 2] * X[:, 3]], axis=1).astype(np.float32)
    net = EnsembleMLP(6, 2, width=528, hidden=2, members=2, batch=32, seed=5)
    net.fit_normalization(X, Y)
    hist = net.train(X, Y, epochs=30, lr=1e-3)
    print("loss", hist[0], hist[-1], flush=True)
    assert np.all(hist[-1] < 0.2 * hist[0])
