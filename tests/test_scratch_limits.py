"""What the library's host code does when device memory runs out: the call
reports it, and the next call that fits neither uses freed or missing arrays
nor is refused; and what the creation of a small context costs in calls of the
runtime.  On the CPU, over a HIP runtime without a device (fake_hip.cpp) whose
allocations fail from a given size on; each case runs in a process of its own,
since the library binds to one runtime."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes as C, sys
sys.path.insert(0, {root!r})
hip = C.CDLL({fake!r}, mode=C.RTLD_GLOBAL)
hip.fake_allocated.restype = C.c_size_t
hip.fake_live.restype = C.c_size_t
hip.fake_fail_above.argtypes = hip.fake_capacity.argtypes = [C.c_size_t]
ANY = 2**64 - 1
import numpy as np
import netflux_amd as nf
from netflux_amd.mlp import Mlp

def fails(call):
    try:
        call()
    except RuntimeError as e:
        assert "out of memory" in str(e), e
        return True

def allocates(call):
    before = hip.fake_allocated()
    call()
    return hip.fake_allocated() - before
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    fake = tmp_path_factory.mktemp("fake_hip") / "fake_hip.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", fake, os.path.join(HERE, "fake_hip.cpp")],
                   check=True)

    def go(body):
        code = PRELUDE.format(root=os.path.dirname(HERE), fake=str(fake)) + body
        p = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
        assert p.returncode == 0, p.stderr

    return go


def test_failure_is_reported_once(run):
    """The runtime keeps the error of a failed allocation; a launch of the next
    call must not find it."""
    run("""
net = Mlp(1)
hip.fake_fail_above(50 << 20)
assert fails(lambda: net.predict(np.ones((3000000, 6), np.float32)))
net.predict(np.ones((256, 6), np.float32))
from tests.mixed_meshes import mixed_box
cfg = nf.Config(density_fs=1.0, pressure_fs=0.7, check_physical_validity=False)
for mesh in (nf.Mesh.box(3), mixed_box((2, 2, 2))):
    s = nf.EulerSolver(cfg, mesh)
    U = s.get_solver_data().get_solution()
    s.set_state(U)
    hip.fake_fail_above(100 << 10)
    assert fails(lambda: s.run(100000))  # its history of 800 KB
    hip.fake_fail_above(ANY)
    s.set_state(U)
""")


def test_network_workspace_that_could_not_grow(run):
    run("""
net = Mlp(1)
x, y = np.ones((300000, 6), np.float32), np.ones((300000, 5), np.float32)
net.loss_grad(x[:256], y[:256])
hip.fake_fail_above(100 << 20)  # the 154 MB arrays of the larger batch
assert fails(lambda: net.loss_grad(x, y))
hip.fake_fail_above(ANY)
# the arrays of the first call went to make room
assert allocates(lambda: net.loss_grad(x[:256], y[:256])) > 128 * 256 * 4 * 3
assert allocates(lambda: net.loss_grad(x[:256], y[:256])) == 0
""")


@pytest.mark.parametrize("now,then,limit", [("mixed", "fp64", 4 << 20), ("fp64", "mixed", 2 << 20)])
def test_precision_switch_without_room(run, now, then, limit):
    # 48,000 cells: the new precision's primvars (1.9 or 1 MB) fit, its face values (7.7 or 3.8 MB) do not
    run(f"""
cfg = nf.Config(density_fs=1.0, pressure_fs=0.7, precision={now!r})
s = nf.EulerSolver(cfg, nf.Mesh.box(20))
hip.fake_fail_above({limit})
for _ in range(2):
    assert fails(lambda: s.set_precision({then!r}))
hip.fake_fail_above(ANY)
assert allocates(lambda: s.set_precision({then!r})) > {limit}
assert allocates(lambda: (s.set_precision({now!r}), s.set_precision({then!r}))) == 0
""")


def test_context_without_room_for_the_face_tables(run):
    """The tables of the sweeps over block faces are what a context can do
    without: one that fits only without them is made all the same, and every
    array made with a context comes before them."""
    run("""
cfg = nf.Config(density_fs=1.0, pressure_fs=0.7, check_physical_validity=True, local_time_step=True)
mesh = nf.Mesh.box(20)
first = nf.Config(density_fs=1.0, pressure_fs=0.7, check_physical_validity=True, local_time_step=True, spatial_order="First")
import gc
def made(c):
    s = nf.EulerSolver(c, mesh)
    n = hip.fake_live()
    del s
    gc.collect()
    assert hip.fake_live() == 0
    return n
full, least = made(cfg), made(first)  # (first order has no use for the tables)
assert full - least > 24 * mesh.n_cells
hip.fake_capacity(full - 1)
assert made(cfg) < full
hip.fake_capacity(least)
assert made(cfg) == least
hip.fake_capacity(least - 1)
try:
    made(cfg)
except RuntimeError:
    sys.exit(0)
sys.exit("a context without room for its arrays was made")
""")


def test_host_steps_without_pinned_memory(run):
    """The pinned record of a host-driven step's results, and the pinned pieces
    of large copies, are what a context can do without."""
    run("""
from tests.mixed_meshes import mixed_box
hip.fake_fail_host(1)
cfg = nf.Config(density_fs=1.0, pressure_fs=0.7)
cfg.delta_time = 1e-3
for mesh in (nf.Mesh.box(3), nf.Mesh.box(24), mixed_box((3, 2, 2))):
    s = nf.EulerSolver(cfg, mesh)
    U = s.get_solver_data().get_solution()
    for _ in range(2):
        s.set_state(U)
        s.step(cfg)
""")


def test_runtime_calls_of_a_small_context(run):
    """Without the tables of the sweeps over block faces a context took 41
    allocations and 31 waits, most of the time that a small one takes to make."""
    run("""
s = nf.EulerSolver(nf.Config(density_fs=1.0, pressure_fs=0.7), nf.Mesh.box(6))
assert hip.fake_allocations() <= 41, hip.fake_allocations()
assert hip.fake_waits() <= 31, hip.fake_waits()
""")


def test_failed_creation_gives_everything_back(run):
    """A context or network that does not fit leaves no device memory behind,
    so that a smaller one fits where it would have without the attempt."""
    run("""
import gc
from tests.mixed_meshes import mixed_box
cfg = nf.Config(density_fs=1.0, pressure_fs=0.7)
def creation_fails(make):
    try:
        make()
    except RuntimeError:
        return True
for large, small in ((nf.Mesh.box(20), nf.Mesh.box(5)), (mixed_box((12, 12, 12)), mixed_box((3, 3, 3)))):
    s = nf.EulerSolver(cfg, large)
    need = hip.fake_live()
    del s
    gc.collect()
    for part in (0.2, 0.5, 0.9):  # fails early, halfway and late
        hip.fake_capacity(int(part * need))
        assert creation_fails(lambda: nf.EulerSolver(cfg, large))
        gc.collect()
        assert hip.fake_live() == 0, (part, hip.fake_live())
    s = nf.EulerSolver(cfg, small)
    del s
    gc.collect()
    hip.fake_capacity(ANY)
hip.fake_capacity(100000)
assert creation_fails(lambda: Mlp(1))
assert hip.fake_live() == 0
""")
