"""Host-driven steps read the run state that the step's last kernel left in
host memory: every call that changes the state on the device in between has to
be seen by the next one."""
import numpy as np
import pytest

import netflux_amd as nf
from tests.cases import pulse_state, sod_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [dict(), dict(precision="mixed"), dict(check_physical_validity=True)])
def test_state_seen_between_calls(kw):
    print(f"[case] host steps {kw}", flush=True)
    mesh = nf.Mesh.box((6, 5, 4), jitter=0.1, patches=("SlipWall",) * 6)
    cfg = sod_config(rk3_zero_old_first_step=False, **kw)
    U = pulse_state(mesh, mach=0.0)
    s, ref = nf.EulerSolver(cfg, mesh), nf.EulerSolver(cfg, mesh)

    def host(n):
        for _ in range(n):
            s.calc_timestep(cfg)
            s.step(cfg)

    s.set_state(U, U)
    ref.set_state(U, U)
    host(2)
    assert len(s.residuals()) == 2
    s.run(3, check_every=3)
    assert len(s.residuals()) == 5
    host(1)
    ref.run(6, check_every=2)
    np.testing.assert_array_equal(s.residuals(), ref.residuals())
    np.testing.assert_array_equal(s.get_solver_data().get_solution(), ref.get_solver_data().get_solution())
    # a state without physical meaning (its steps may raise), and the next one
    bad = U.copy()
    bad[7, 4] = -1.0
    s.set_state(bad, bad)
    try:
        host(3)
    except RuntimeError:
        pass
    s.set_state(U, U)
    assert len(s.residuals()) == 0
    s.eval_flux_balance()
    host(1)
    assert len(s.residuals()) == 1
    np.testing.assert_array_equal(s.residuals(), ref.residuals()[:1])


def test_many_contexts_alive():
    """More contexts than a page of pinned records holds, stepped in turn and
    given back out of order; new ones take the freed records."""
    print("[case] host steps of 40 contexts", flush=True)
    mesh = nf.Mesh.box((3, 2, 2), patches=("SlipWall",) * 6)
    hexes = nf.Mesh.hex_box(2, patches=("SlipWall",) * 6)
    out = {}
    for m in (mesh, hexes):
        cfg = sod_config(rk3_zero_old_first_step=False)
        U = pulse_state(m, mach=0.0)
        live = [nf.EulerSolver(cfg, m) for _ in range(40)]
        for s in live:
            s.set_state(U, U)
        for _ in range(2):
            for s in live:
                s.calc_timestep(cfg)
                s.step(cfg)
        del live[::2], s
        again = nf.EulerSolver(cfg, m)
        again.set_state(U, U)
        for _ in range(2):
            again.calc_timestep(cfg)
            again.step(cfg)
        for s in live:
            np.testing.assert_array_equal(s.get_solver_data().get_solution(), again.get_solver_data().get_solution())
            np.testing.assert_array_equal(s.residuals(), again.residuals())
