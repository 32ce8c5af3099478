"""Uploads on either side of the size from which they go through pinned pieces
(32 MiB): every sample of a host array arrives, seen from the outputs of a few
that are sent by themselves."""
import numpy as np
import pytest

from tests.test_zz_no_alloc import _features, _net

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(32 << 20) // 24, (32 << 20) // 24 + 1, 1500007])
def test_inputs_around_the_limit(n):
    print(f"[case] upload of {24 * n} bytes", flush=True)
    net = _net(seed=3)
    x = _features(n, 4)
    y = net.predict(x)
    assert np.isfinite(y).all()
    pick = np.r_[0:3, n // 2 - 1:n // 2 + 2, n - 3:n]
    np.testing.assert_array_equal(net.predict(x[pick]), y[pick])
    np.testing.assert_array_equal(net.predict(x[n - 9000:]), y[n - 9000:])
