"""Training kernels at the edges of their tiles -- 16 samples per tile, rows
padded to 64, batch splits of 512, more tiles than blocks -- against the
rounding-emulating FP64 restatement of the network."""
import numpy as np
import pytest

from oracle import mlp_ref as M
from tests.test_gpu_mlp import _data, _net

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 511, 512, 513, 1088, 4096, 4113])
def test_loss_and_gradient_at_tile_edges(n):
    print(f"[case] training kernels n={n}", flush=True)
    net, p, (sh, sc, osh, osc) = _net(seed=4)
    x, y = _data(n, seed=n)
    loss, g = net.loss_grad(x, y)
    tn = ((y - osh) * (np.float32(1) / osc)).astype(np.float64)
    loss_ref, g_ref = M.loss_grad(p.astype(np.float32), M.normalise_inputs(x, sh, sc), tn, emulate=True)
    assert abs(loss - loss_ref) <= 1e-4 * loss_ref
    # FP32 accumulation, and now and then an activation one BF16 ulp (2^-8)
    # off: 2^-8 / sqrt(128) = 3.5e-4 of a block's gradient for one sample
    for a, b in zip(M.unpack(g), M.unpack(g_ref)):
        assert np.linalg.norm(a - b) <= 5e-3 * np.linalg.norm(b)
    # the same call again, after a larger one: no stale padding
    net.loss_grad(*_data(n + 700, seed=1))
    loss2, g2 = net.loss_grad(x, y)
    assert loss2 == loss
    np.testing.assert_array_equal(g2, g)
