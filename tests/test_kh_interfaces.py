"""The batched Kelvin-Helmholtz interfaces are the per-sample ones bit for
bit: blocks of one sample and of many, odd sizes, a zero amplitude sum."""
import numpy as np
import pytest

from alsvinn_amd.initial_data import kh_interfaces, kh_interfaces_many


@pytest.mark.parametrize("n,samples", [(1, 2), (7, 3), (33, 300), (128, 4), (512, 16), (4099, 3)])
def test_batched_interfaces_bitwise(n, samples):
    p = np.random.default_rng(n).random((samples, 40))
    p[1, :10] = 0.0
    want = np.stack([np.stack(kh_interfaces(n, row)) for row in p])
    got = kh_interfaces_many(n, p)
    np.testing.assert_array_equal(got.view(np.uint64), want.view(np.uint64))
