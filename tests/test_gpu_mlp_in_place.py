"""nf_mlp_predict_noalloc with outputs over its inputs, as a serving loop with
one buffer calls it: every block's inputs have to be read before any output
replaces them.  Against nf_mlp_predict, bit for bit, on a stream of the
caller's; y before, on and behind the start of x, and just past its end."""
import ctypes as C

import numpy as np
import pytest
import torch

from netflux_amd import _abi as A
from tests.test_zz_no_alloc import _features, _net

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 17, 777, 12289, 16384])
def test_outputs_over_inputs(n):
    net = _net(seed=7)
    x = _features(n, n)
    ref = net.predict(x)
    s = torch.cuda.Stream()
    for off in (0, -4, 3, 2 * n, 6 * n - 1, 6 * n):  # floats from x to y
        print(f"[case] predict in place n={n} offset={off}", flush=True)
        buf = torch.full((12 * n + 64,), float("nan"), device="cuda")
        xd, yd = buf[8:8 + 6 * n], buf[8 + off:8 + off + 5 * n]
        xd.copy_(torch.from_numpy(x.ravel()))
        torch.cuda.synchronize()
        rc = A.lib().nf_mlp_predict_noalloc(net._h, C.c_void_p(xd.data_ptr()), n, C.c_void_p(yd.data_ptr()),
                                            C.c_void_p(s.cuda_stream))
        assert rc == A.NF_OK
        s.synchronize()
        np.testing.assert_array_equal(yd.cpu().numpy().reshape(n, 5), ref)
