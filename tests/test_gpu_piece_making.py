"""Downloads of a context that meets a pool without pinned pieces: a first one
that is too small to make them, a second that makes them, one that finds
them, and one that makes them at once by its size."""
import gc

import numpy as np
import pytest

import netflux_amd as nf
from tests.cases import pulse_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(20, 21, 22), (52, 52, 52)])  # 2.2 and 33.7 MB of state
def test_downloads_of_a_lone_context(n):
    print(f"[case] lone context {n}", flush=True)
    mesh = nf.Mesh.box(n)
    cfg = pulse_config(spatial_order="First")
    for life in range(2):
        gc.collect()
        s = nf.EulerSolver(cfg, mesh)
        for seed in range(3):
            U = np.random.default_rng(seed).random((s.N, 5)) + 1.0
            s.set_state(U)
            np.testing.assert_array_equal(s.get_solver_data().get_solution(), U)
        del s
