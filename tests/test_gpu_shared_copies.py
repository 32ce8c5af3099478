"""State transfers of several contexts at once: from the fifth user on, plain
copies of 256 KiB and more go through one stream of the pool, while larger
downloads borrow pinned pieces.  Every context gets its own state back, in one
thread and in several, also after the others have gone."""
import gc
import threading

import numpy as np
import pytest

import netflux_amd as nf
from tests.cases import pulse_config

pytestmark = pytest.mark.gpu

# cells x 40 bytes: under and over 256 KiB, under and over 2 MiB
SIZES = [(3, 2, 2), (12, 13, 7), (10, 11, 10), (16, 17, 32), (17, 18, 29), (30, 20, 21)]


def _contexts(n):
    cfg = pulse_config(rk3_zero_old_first_step=False)
    return [nf.EulerSolver(cfg, nf.Mesh.box(SIZES[i % len(SIZES)])) for i in range(n)]


def _round_trips(s, seed, times, bad):
    r = np.random.default_rng(seed)
    for _ in range(times):
        U = r.random((s.N, 5)) + 1.0
        s.set_state(U)
        if not np.array_equal(s.get_solver_data().get_solution(), U):
            bad.append(s.N)


@pytest.mark.parametrize("users", [1, 4, 5, 12])
def test_every_context_gets_its_own_state(users):
    print(f"[case] {users} contexts, one thread", flush=True)
    ctx = _contexts(users)
    U = [np.random.default_rng(i).random((s.N, 5)) + 1.0 for i, s in enumerate(ctx)]
    for _ in range(3):
        for s, u in zip(ctx, U):
            s.set_state(u)
        for s, u in reversed(list(zip(ctx, U))):
            np.testing.assert_array_equal(s.get_solver_data().get_solution(), u)
    # a step between, and the pool's stream gone with all users but one
    last, u = ctx[-1], U[-1]
    ctx.clear()
    gc.collect()
    last.set_state(u)
    last.run(1)
    assert not np.array_equal(last.get_solver_data().get_solution(), u)
    last.set_state(u)
    np.testing.assert_array_equal(last.get_solver_data().get_solution(), u)


def test_threads_of_contexts():
    print("[case] 12 contexts, 12 threads", flush=True)
    bad = []
    threads = [threading.Thread(target=_round_trips, args=(s, i, 20, bad)) for i, s in enumerate(_contexts(12))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
