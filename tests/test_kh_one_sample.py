"""A batch of one sample gets kh_interfaces' bits too, and is taken by itself."""
import numpy as np
import pytest

from alsvinn_amd import initial_data


@pytest.mark.parametrize("n", [1, 16, 64, 1000, 4099])
def test_lone_sample_bitwise(n, monkeypatch):
    p = np.random.default_rng(n).random((1, 40))
    p[0, 10:20] *= n != 16
    want = np.stack(initial_data.kh_interfaces(n, p[0]))
    calls = []
    one = initial_data.kh_interfaces
    monkeypatch.setattr(initial_data, "kh_interfaces", lambda *a: calls.append(a) or one(*a))
    got = initial_data.kh_interfaces_many(n, p)
    assert got.shape == (1, 2, n) and len(calls) == 1
    np.testing.assert_array_equal(got[0].view(np.uint64), want.view(np.uint64))
