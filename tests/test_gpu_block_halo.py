"""Second-order sweeps over blocks that gather their halo once and evaluate
their faces once, against the oracle bit for bit: blocks without a halo,
ragged last blocks, halos of more than one round of lanes, and cells without
locality, whose halos do not fit and which are gathered per lane; and the
options of a step against the sweeps that gather per lane."""
import numpy as np
import pytest

import netflux_amd as nf
from tests.cases import pulse_config, pulse_state, sod_config
from tests.oracle_bind import Oracle

pytestmark = pytest.mark.gpu


def _shuffled(n, seed, patches=("SlipWall", "NoSlipWall") * 3):
    m = nf.Mesh.box(n, jitter=0.15 if min(n) > 1 else 0.0, patches=patches)
    nodes, cells, pn, pf, pbc = m.arrays()
    first = np.concatenate([[0], np.cumsum(pn.astype(np.int64))])
    cells = cells[np.random.default_rng(seed).permutation(len(cells))]
    return nf.Mesh.from_arrays(nodes, cells, [pf[first[i]:first[i + 1]] for i in range(len(pn))], list(pbc))


@pytest.mark.parametrize("n,order,limiter", [
    ((1, 1, 1), "morton", "Barth"),     # 6 cells, no outside neighbour
    ((6, 7, 1), "morton", "NONE"),      # 252 cells: one ragged block, boundary entries only
    ((11, 2, 2), "rcm", "Barth"),       # 264: eight cells in the last block
    ((60, 2, 3), "input", "NONE"),      # slabs: long halos
    ((13, 12, 11), "morton", "Barth"),
    ((13, 12, 11), "input", "Barth"),   # shuffled and kept so: nearly every neighbour outside
    ((9, 8, 7), "input", "NONE"),
])
def test_matches_oracle(n, order, limiter):
    print(f"[case] block halos {n} {order} {limiter}", flush=True)
    mesh = _shuffled(n, 5)
    cfg = sod_config(limiter=limiter, cell_order=order, rk3_zero_old_first_step=False)
    g, o = nf.EulerSolver(cfg, mesh), Oracle.from_mesh(mesh, cfg)
    U = pulse_state(mesh, mach=0.0)
    g.set_state(U, U)
    o.set_state(U, uold_equals_u=True)
    g.calc_timestep(cfg)
    assert cfg.delta_time == o.calc_timestep()
    g.step(cfg)
    o.step(cfg.delta_time)
    g.run(6, check_every=3)
    o.run(6)
    np.testing.assert_array_equal(g.get_solver_data().get_solution(), o.get("U"))


@pytest.mark.parametrize("kw", [
    dict(inv_flux="HLLC"), dict(limiter="NONE", inv_flux="HLLC"), dict(local_time_step=True),
    dict(check_physical_validity=True), dict(time_scheme="ExplicitEuler", limiter="NONE")])
def test_equals_the_gathering_sweeps(kw):
    """256-cell blocks (block faces) against 128-cell blocks (per lane), on a
    farfield mesh of nine blocks, also a batch's second instance; the fields
    of an evaluation as well."""
    kw = dict(kw)
    flux = kw.pop("inv_flux", "Rusanov")
    print(f"[case] block faces {kw} {flux}", flush=True)
    mesh = _shuffled((8, 7, 6), 3, ("FarField", "SlipWall", "NoSlipWall") * 2)
    cfg = pulse_config(inviscid_flux_scheme=flux, rk3_zero_old_first_step=False, **kw)
    U = pulse_state(mesh)
    out = []
    for block in (256, 128):
        g = nf.EulerSolver(cfg, mesh)
        g.set_launch(block)
        g.set_state(U, U)
        g.run(7, check_every=3)
        g.eval_flux_balance()
        d = g.get_solver_data()
        b = nf.BatchSolver(cfg, [nf.Mesh.box((3, 2, 1)), mesh])
        b.set_launch(block)
        b.set_state(1, U, U)
        b.run(7, check_every=3)
        np.testing.assert_array_equal(b.get_solution(1), d.get_solution())
        out.append([d.get_solution(), d.get_flux_balance(), d.get_primvars_gradient(), d.get_primvars_limiter()])
    for a, b in zip(*out):
        assert np.isfinite(a).all()
        np.testing.assert_array_equal(a, b)
