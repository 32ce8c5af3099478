"""Host arrays across the boundary, on both sides of the size from which they
go through pinned pieces (2 MiB) and of a piece (4 MiB): a round trip of the
state returns its bits, also from and into arrays that start anywhere, and
inference gives every sample its own result."""
import ctypes as C

import numpy as np
import pytest

import netflux_amd as nf
from netflux_amd import _abi as A
from tests.cases import pulse_config
from tests.test_gpu_mlp import _data, _net

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(20, 20, 21), (20, 20, 22), (30, 30, 20), (47, 31, 29), (53, 47, 41)])
@pytest.mark.parametrize("kind", ["tet", "hex"])
def test_state_round_trip(n, kind):
    print(f"[case] state round trip {kind} {n}", flush=True)
    if kind == "hex":
        n = (n[0] * 6, n[1], n[2])
        if n[0] * n[1] * n[2] > 150000:
            pytest.skip("as the tetrahedral case of that size")
    mesh = nf.Mesh.box(n) if kind == "tet" else nf.Mesh.hex_box(n)
    s = nf.EulerSolver(pulse_config(rk3_zero_old_first_step=False), mesh)
    rng = np.random.default_rng(n[0])
    raw = np.empty(8 * 5 * s.N + 5, np.uint8)
    for off in (0, 5):  # (numpy wants aligned doubles: the odd address goes through the C ABI)
        U = rng.random((s.N, 5)) + 1.0
        raw[off:off + U.nbytes] = U.view(np.uint8).ravel()
        p = raw.ctypes.data + off
        assert A.lib().nf_set_state(s._ctx, C.cast(p, A.f64p), C.cast(p, A.f64p)) == A.NF_OK
        np.testing.assert_array_equal(s.get_solver_data().get_solution(), U)
        raw[:] = 0
        assert A.lib().nf_get_state(s._ctx, C.cast(p, A.f64p)) == A.NF_OK
        np.testing.assert_array_equal(raw[off:off + U.nbytes], U.view(np.uint8).ravel())


def test_old_state_must_equal_state():
    print("[case] U_old given", flush=True)
    s = nf.EulerSolver(pulse_config(rk3_zero_old_first_step=False), nf.Mesh.box(4))
    U = np.random.default_rng(0).random((s.N, 5)) + 1.0
    s.set_state(U, U)
    s.set_state(U, U.copy())
    V = U.copy()
    V[-1, 4] += 1e-9
    with pytest.raises(RuntimeError, match="U_old must be NULL"):
        s.set_state(U, V)


@pytest.mark.parametrize("n", [87381, 87382, 104857, 104858, 300007])
def test_predict_sizes(n):
    print(f"[case] predict host arrays n={n}", flush=True)
    net = _net(seed=2)[0]
    x, _ = _data(n, seed=3)
    y = net.predict(x)
    pick = np.r_[0:3, n // 2:n // 2 + 3, n - 3:n]
    np.testing.assert_array_equal(net.predict(x[pick]), y[pick])
