"""Second-order sweeps over blocks that gather their halo once, against the
oracle bit for bit: blocks without a halo, ragged last blocks, halos of more
than one round of lanes, and cells without locality, whose halos do not fit
and which are gathered per lane."""
import numpy as np
import pytest

import netflux_amd as nf
from tests.cases import pulse_state, sod_config
from tests.oracle_bind import Oracle

pytestmark = pytest.mark.gpu


def _shuffled(n, seed):
    m = nf.Mesh.box(n, jitter=0.15 if min(n) > 1 else 0.0, patches=("SlipWall", "NoSlipWall") * 3)
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
