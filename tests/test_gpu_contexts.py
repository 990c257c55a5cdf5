"""Solvers, batches, statistics and networks whose context is destroyed before
them: they go on working, and both orders of destruction leave the device
usable.  Their pinned memory is the context's pool, which has to live as long as
the last of them (the pool itself: test_pinned_pool.py)."""
import numpy as np
import pytest

import alsvinn_amd
from alsvinn_amd import BatchRunner, Simulator, _abi
from alsvinn_amd.surrogate import EnsembleMLP
from alsvinn_amd.uq import MeanVariance
from tests.cases import smooth_state

pytestmark = pytest.mark.gpu

N = (40, 24, 1)


class _OwnContext:
    """Objects made inside take a context of their own, which goes at the end
    of the block, before them."""

    def __enter__(self):
        self.saved = dict(alsvinn_amd.simulator._default_ctx)
        alsvinn_amd.simulator._default_ctx.clear()
        self.ctx = alsvinn_amd.simulator.default_context()
        return self.ctx

    def __exit__(self, *a):
        _abi.check(_abi.load().avh_ctx_destroy(self.ctx._h))
        self.ctx._h = None
        alsvinn_amd.simulator._default_ctx.clear()
        alsvinn_amd.simulator._default_ctx.update(self.saved)


def _sim(n=N):
    s = Simulator("euler2", "weno2", "hll3", "rungekutta3", "periodic", n, cfl=0.4)
    s.set_interior(smooth_state("euler2", n[:2], seed=4))
    return s


def _batch():
    br = BatchRunner("euler2", "weno2", "hll3", "rungekutta3", "periodic", [(N, 3)], 0.02, cfl=0.4, stats_saves=1)
    for k in range(3):
        br.set_state(0, k, smooth_state("euler2", N[:2], seed=4))
    return br


def test_context_goes_first():
    print("case contexts", flush=True)
    want = _sim()
    want.run(0.02)
    want_batch = _batch()
    want_batch.run(chunk=8)
    with _OwnContext():
        got = [_sim() for _ in range(70)]  # more than the pool's page holds
        br = _batch()
        st = MeanVariance("euler2", N)
        net = EnsembleMLP(3, 2, width=16, hidden=1, members=1, batch=16, seed=1)
    for s in (got[0], got[69]):
        s.run(0.02)
        np.testing.assert_array_equal(s.get_interior(), want.get_interior())
    br.run(chunk=8)
    for k in range(3):
        np.testing.assert_array_equal(br.get_state(0, k), want_batch.get_state(0, k))
    st.accumulate(got[0])
    np.testing.assert_array_equal(st.read()[0], want.get_interior())
    X = np.random.default_rng(0).random((32, 3)).astype(np.float32)
    a = net.predict_members(X)
    net.train(X, X[:, :2], epochs=1)
    assert np.isfinite(a).all() and np.isfinite(net.get_params(0)).all()
    del got, br, st, net, s
    again = _sim()
    again.run(0.02)
    np.testing.assert_array_equal(again.get_interior(), want.get_interior())


def test_solver_goes_first():
    with _OwnContext():
        s = _sim()
        s.run(0.01)
        at = s.get_current_time()
        del s
    again = _sim()
    again.run(0.01)
    assert again.get_current_time() == at
