"""Reductions of a batch whose meshes have different numbers of chunks (2,048
sweep blocks each): one mesh of two chunks among meshes of one, one of them
stopped by its drop.  Residuals, time steps and states have to be those of
each mesh alone, bit for bit, and the two-chunk residuals those of one chunk
(256-cell blocks) up to the order of the sum."""
import numpy as np
import pytest

import netflux_amd as nf
from tests.cases import pulse_config, pulse_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("where", [0, 1, 2])
def test_batch_with_a_mesh_of_two_chunks(where):
    print(f"[case] two chunks at instance {where}", flush=True)
    cfg = pulse_config(rk3_zero_old_first_step=False)
    sizes = [(6, 5, 4), (9, 8, 7)]
    sizes.insert(where, (36, 35, 35))  # 264,600 cells: 2,068 blocks of 128, 1,034 of 256
    stopped = 2 if where < 2 else 0
    meshes = [nf.Mesh.box(n, jitter=0.1, patches=("FarField", "SlipWall", "NoSlipWall") * 2) for n in sizes]
    states = [pulse_state(m) for m in meshes]
    b = nf.BatchSolver(cfg, meshes)
    b.set_launch(128)
    for i, U in enumerate(states):
        b.set_state(i, U)
    b.set_residual_ref(stopped, 1e30)  # converges in its first step
    stats = b.run(4, residual_drop=1e-9, check_every=2)
    for i, (m, U) in enumerate(zip(meshes, states)):
        n = 1 if i == stopped else 4
        assert len(b.residuals(i)) == n
        for block in (128, 256) if i == where else (128,):
            g = nf.EulerSolver(cfg, m)
            g.set_launch(block)
            g.set_state(U)
            one = g.run(n, check_every=2)
            assert (stats[i]["time"], stats[i]["last_dt"]) == (one["time"], one["last_dt"])
            np.testing.assert_array_equal(b.get_solution(i), g.get_solver_data().get_solution())
            # sums of non-negative terms, about 25 additions deep either way: 25 eps before the square root
            np.testing.assert_allclose(b.residuals(i), g.residuals(), rtol=0 if block == 128 else 1e-14, atol=0)
