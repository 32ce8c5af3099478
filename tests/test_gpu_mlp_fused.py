"""The fused inference kernel at the edges of its sample tiles (16 and 64 per
block) and of the rule between them, against the FP64 restatement of the
network with BF16 rounding at the device's rounding points."""
import ctypes as C

import numpy as np
import pytest

from netflux_amd import _abi as A
from oracle import mlp_ref as M
from tests.test_gpu_mlp import _data, _net
from tests.test_zz_no_alloc import DevBuf, _hip

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


def test_device_calls_overlap_on_two_streams():
    """nf_mlp_predict_noalloc calls of two networks, in turn on two streams
    without waiting between them, share nothing: each gives its own result."""
    print("[case] fused predict, two networks on two streams", flush=True)
    hip = _hip()
    nets = [_net(seed=11)[0], _net(seed=12)[0]]
    xs = [_data(700, seed=21 + q)[0] for q in range(2)]
    ref = [n.predict(x) for n, x in zip(nets, xs)]
    streams = [C.c_void_p(), C.c_void_p()]
    bufs = [(DevBuf(hip, x.nbytes), DevBuf(hip, len(x) * 20)) for x in xs]
    try:
        for s in streams:
            assert hip.hipStreamCreate(C.byref(s)) == 0  # default priority
        for x, (xd, yd) in zip(xs, bufs):
            xd.put(x)
            yd.put(np.full((len(x), 5), np.nan, np.float32))
        for _ in range(20):
            for net, s, x, (xd, yd) in zip(nets, streams, xs, bufs):
                assert A.lib().nf_mlp_predict_noalloc(net._h, xd.p, len(x), yd.p, s) == A.NF_OK
        for q, s in enumerate(streams):
            assert hip.hipStreamSynchronize(s) == 0
            np.testing.assert_array_equal(bufs[q][1].get((len(xs[q]), 5)), ref[q])
    finally:
        for xd, yd in bufs:
            xd.free()
            yd.free()
        for s in streams:
            hip.hipStreamDestroy(s)
