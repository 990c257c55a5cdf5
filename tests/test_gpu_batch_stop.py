"""A batch stops launching once its last sample has ended; states, times, step
counts, statistics and the steps reported are those of a run that launches
every step of its chunks, with and without graphs."""
import numpy as np
import pytest

from alsvinn_amd.uq import BatchRunner

pytestmark = pytest.mark.gpu


def _run(chunk, graph_steps, max_steps=1 << 62, t_end=0.02):
    br = BatchRunner("euler2", "weno2", "hll3", "rungekutta3", "periodic", [((24, 24), 5), ((40, 40), 2)], t_end,
                     cfl=0.4, stats_saves=2)
    br.set_graph_steps(graph_steps)
    for g, m in ((0, 5), (1, 2)):
        br.set_kelvin_helmholtz(g, np.random.default_rng(g).random((m, 40)))
    done, left = br.run(max_steps=max_steps, chunk=chunk)
    out = [br.get_state(g, s) for g, m in ((0, 5), (1, 2)) for s in range(m)]
    prog = [(p.time, p.last_dt, p.steps, p.violated) for g, m in ((0, 5), (1, 2))
            for p in (br.progress(g, s) for s in range(m))]
    stats = [br.statistics(g, k) for g in range(2) for k in range(2)]
    return done, left, out, prog, stats


@pytest.mark.parametrize("graph_steps", [0, 3, 8])
def test_early_stop_changes_nothing(graph_steps):
    want = _run(1, 0)
    assert want[1] == 0
    for chunk in (1, 7, 16, 17, 500):
        print("case batch stop", graph_steps, chunk, flush=True)
        got = _run(chunk, graph_steps)
        assert got[1] == 0
        assert got[0] == -(-want[0] // chunk) * chunk
        assert got[3] == want[3]
        for a, b in zip(got[2], want[2]):
            np.testing.assert_array_equal(a.view(np.uint64), b.view(np.uint64))
        for (m, v, c), (mw, vw, cw) in zip(got[4], want[4]):
            assert c == cw
            np.testing.assert_array_equal(m, mw)
            np.testing.assert_array_equal(v, vw)


def test_max_steps_inside_a_graph():
    """max_steps before the end, not a multiple of the graph's steps."""
    want = _run(1, 0, max_steps=27, t_end=0.1)
    got = _run(64, 8, max_steps=27, t_end=0.1)
    assert got[:2] == want[:2] and got[0] == 27 and got[1] > 0
    assert got[3] == want[3]
