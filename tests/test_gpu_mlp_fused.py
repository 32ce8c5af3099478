"""The fused inference kernel at the edges of its sample tiles (16 and 64 per
block) and of the rule between them, against the FP64 restatement of the
network with BF16 rounding at the device's rounding points."""
import numpy as np
import pytest

from oracle import mlp_ref as M
from tests.test_gpu_mlp import _data, _net

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 12287, 12288, 12289, 12353, 65537])
def test_predict_at_tile_edges(n):
    print(f"[case] fused predict n={n}", flush=True)
    net, p, (sh, sc, osh, osc) = _net(seed=9)
    x, _ = _data(n, seed=n)
    y = net.predict(x)
    yn, _ = M.forward(p.astype(np.float32), M.normalise_inputs(x, sh, sc), emulate=True)
    # one BF16 ulp of an activation (2^-8 of about 2) through a weight of at
    # most 1/sqrt(128), a few of them: 2e-3 in normalised units
    assert (np.abs(y - (yn * osc + osh)) / osc).max() < 2e-3
    # samples are independent: the last ones alone give the same bits
    k = min(n, 5)
    np.testing.assert_array_equal(net.predict(x[-k:]), y[-k:])
