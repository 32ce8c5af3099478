"""Boundary ghosts in launches of their own (large contexts) against those
that the sweeps store (small ones): small meshes, one of them with every cell
on the boundary, in a batch with a mesh that takes the separate launches by
itself, have the bits they have alone.  Which way a context takes is seen from
the launches of its step, not from a size."""
import numpy as np
import pytest

import netflux_amd as nf
from tests.cases import pulse_config, pulse_state

pytestmark = pytest.mark.gpu


def _separate(solver):
    return any(name.startswith("ghost_face") for name in solver.time_kernels(1))


@pytest.mark.parametrize("precision,block", [("fp64", 256), ("fp64", 128), ("mixed", 256), ("mixed", 128)])
def test_small_meshes_in_a_batch_with_separate_launches(precision, block):
    print(f"[case] separate vs fused ghosts, {precision}, block {block}", flush=True)
    cfg = pulse_config(precision=precision, rk3_zero_old_first_step=False)
    sizes = [(1, 1, 1), (5, 4, 3), (9, 8, 7)]
    meshes = [nf.Mesh.box(n, jitter=0.1 if min(n) > 1 else 0.0, patches=("FarField", "SlipWall", "NoSlipWall") * 2)
              for n in sizes]
    large = nf.Mesh.box((48, 46, 45), patches=("SlipWall",) * 6)
    alone = nf.EulerSolver(cfg, large)
    alone.set_launch(block)
    assert _separate(alone)  # and so does a batch that has it and more
    b = nf.BatchSolver(cfg, meshes + [large])
    b.set_launch(block)
    for i, m in enumerate(meshes):
        b.set_state(i, pulse_state(m))
    b.run(7, check_every=3)
    for i, m in enumerate(meshes):
        g = nf.EulerSolver(cfg, m)
        g.set_launch(block)
        g.set_state(pulse_state(m))
        g.run(7, check_every=3)
        np.testing.assert_array_equal(b.get_solution(i), g.get_solver_data().get_solution())
        np.testing.assert_array_equal(b.residuals(i), g.residuals())
        assert not _separate(g)
