"""Boundary ghosts at the end of the sweeps (small contexts) against the
oracle and against launches of their own (large contexts): a batch that is
large enough for the separate launches gives each mesh the bits it has alone,
and state changes, stops and precision switches between runs leave no stale
ghosts behind."""
import numpy as np
import pytest

import netflux_amd as nf
from tests.cases import pulse_config, pulse_state, sod_config, sod_state
from tests.oracle_bind import Oracle

pytestmark = pytest.mark.gpu

FUSE_MAX = 1024 * 256  # device cells up to which a context's sweeps store the ghosts


@pytest.mark.parametrize("precision,block", [("fp64", 256), ("fp64", 128), ("mixed", 256), ("mixed", 128)])
def test_batch_with_separate_launches_equals_single(precision, block):
    print(f"[case] fused vs separate ghosts, {precision}, block {block}", flush=True)
    # one tetrahedral block (every cell on the boundary), a ragged box, a box
    # just under the rule alone, over it together
    sizes = [(1, 1, 1), (5, 4, 3), (36, 34, 33)]
    meshes = [nf.Mesh.box(n, jitter=0.1, patches=("FarField", "SlipWall", "NoSlipWall") * 2) for n in sizes]
    assert meshes[2].n_cells < FUSE_MAX < sum(m.n_cells for m in meshes) + 256 * 100
    cfg = pulse_config(precision=precision, rk3_zero_old_first_step=False)
    states = [pulse_state(m) for m in meshes]
    filler = nf.Mesh.box((20, 16, 15), patches=("SlipWall",) * 6)
    b = nf.BatchSolver(cfg, meshes + [filler])
    assert sum(b.N) > FUSE_MAX
    b.set_launch(block)
    for i, U in enumerate(states):
        b.set_state(i, U)
    b.run(7, check_every=3)
    for i, (m, U) in enumerate(zip(meshes, states)):
        g = nf.EulerSolver(cfg, m)
        g.set_launch(block)
        g.set_state(U)
        g.run(7, check_every=3)
        np.testing.assert_array_equal(b.get_solution(i), g.get_solver_data().get_solution())
        np.testing.assert_array_equal(b.residuals(i), g.residuals())


def test_runs_interleaved_with_other_calls():
    """Graph replays, host steps, evaluations, new states and precision
    switches in one context against fresh contexts started from its states."""
    print("[case] fused ghosts, interleaved calls", flush=True)
    mesh = nf.Mesh.box((7, 6, 5), jitter=0.15, patches=("FarField", "SlipWall") * 3)
    cfg = pulse_config(rk3_zero_old_first_step=False)
    g = nf.EulerSolver(cfg, mesh)
    U = pulse_state(mesh)
    g.set_state(U, U)
    for call in ("run", "host", "eval", "run", "precision", "set", "run", "host", "run"):
        U = g.get_solver_data().get_solution()
        if call == "run":
            g.run(6, check_every=2)
        elif call == "host":
            g.calc_timestep(cfg)
            g.step(cfg)
        elif call == "eval":
            g.eval_flux_balance()
            continue
        elif call == "precision":
            g.set_precision("mixed")
            g.run(2, check_every=1)
            g.set_precision("fp64")
            continue
        else:
            U = sod_state(mesh)
            g.set_state(U, U)
            continue
        dt = g.run(0)["last_dt"]
        # a step by hand from U with the dt the context holds: one flux balance each, from a fresh context
        h = nf.EulerSolver(cfg, mesh)
        h.set_state(g.get_solver_data().get_solution(), g.get_solver_data().get_solution())
        c2 = pulse_config(rk3_zero_old_first_step=False)
        c2.delta_time = dt
        h.step(c2)
        g.calc_timestep(cfg)
        assert cfg.delta_time == dt
        g.step(cfg)
        np.testing.assert_array_equal(g.get_solver_data().get_solution(), h.get_solver_data().get_solution())


def test_stopped_instance_runs_again():
    """An instance that reached its drop stays stopped while the others go
    on and take new states; cleared, it continues from its own state."""
    print("[case] fused ghosts, stopped instance", flush=True)
    meshes = [nf.Mesh.box((4, 4, 4), jitter=0.1, patches=("FarField",) * 6) for _ in range(2)]
    cfg = pulse_config(rk3_zero_old_first_step=False)
    U = [pulse_state(meshes[0]), pulse_state(meshes[1], amp=0.05)]
    b = nf.BatchSolver(cfg, meshes)
    for i in (0, 1):
        b.set_state(i, U[i], U[i])
    b.set_residual_ref(0, 1e30)  # instance 0 converges in its first step
    b.run(4, residual_drop=1e-3, check_every=1)
    b.set_state(1, U[1], U[1])
    b.run(3, residual_drop=1e-3, check_every=3)
    b.run(5, check_every=5)
    one = nf.EulerSolver(cfg, meshes[0])
    one.set_state(U[0], U[0])
    one.run(6, check_every=3)
    np.testing.assert_array_equal(b.get_solution(0), one.get_solver_data().get_solution())


@pytest.mark.parametrize("n", [(1, 1, 1), (3, 1, 1), (8, 7, 6)])
def test_wall_boxes_match_oracle(n):
    print(f"[case] fused ghosts vs oracle {n}", flush=True)
    mesh = nf.Mesh.box(n, jitter=0.0 if min(n) < 2 else 0.15)
    cfg = sod_config()
    U = sod_state(mesh)
    g, o = nf.EulerSolver(cfg, mesh), Oracle.from_mesh(mesh, cfg)
    g.set_state(U)
    o.set_state(U)
    g.run(12, check_every=4)
    o.run(12)
    np.testing.assert_array_equal(g.get_solver_data().get_solution(), o.get("U"))


@pytest.mark.parametrize("precision,block", [("fp64", 256), ("fp64", 128), ("mixed", 256)])
def test_large_batch_equals_single(precision, block):
    """The ghosts in launches of their own: a batch of 1,800 blocks against
    its meshes alone, whose sweeps store them."""
    print(f"[case] separate ghosts, {precision}, block {block}", flush=True)
    mesh = nf.Mesh.box((36, 34, 33), jitter=0.1, patches=("FarField", "SlipWall", "NoSlipWall") * 2)
    cfg = pulse_config(precision=precision, rk3_zero_old_first_step=False)
    b = nf.BatchSolver(cfg, [mesh, nf.Mesh.box((34, 33, 33), patches=("SlipWall",) * 6)])
    assert sum(b.N) > 1700 * 256
    U = pulse_state(mesh)
    g = nf.EulerSolver(cfg, mesh)
    for s in (b, g):
        s.set_launch(block)
        s.set_state(*((0, U) if s is b else (U,)))
        s.run(5, check_every=2)
    np.testing.assert_array_equal(b.get_solution(0), g.get_solver_data().get_solution())
    np.testing.assert_array_equal(b.residuals(0), g.residuals())
