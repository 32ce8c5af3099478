"""Workloads whose speed matters to users of netflux_amd, as data.

listed() gives the fixed cases, draw(rng) another case of the same ranges;
prepare / run / work / exact act on one case.  A case is a flat dict:

  kind    what is called (the functions named run_<kind> below)
  n*, k   mesh size: n0 x n1 x n2 hexahedral blocks, or (5k, 2k, k) for a channel
  others  the options of netflux_amd.Config and of the call

Meshes are made here (and given to the library as arrays), so that exact()
can restate the whole path -- face graph, geometry, scheme -- in plain torch
FP64 from the same nodes and cells.
"""
import functools
import math
import os

import numpy as np
import torch

import netflux_amd as nf
from netflux_amd import _abi, steady
from netflux_amd.mlp import Mlp, param_slices

GAMMA = 1.4
NETWORK = "netflux_amd/data/warm_start_bump_512.npz"
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


# ---------------------------------------------------------------------------
# the cases
def listed():
    box = dict(kind="solve", mesh="tet", bc="FarField", jitter=0.15, mode="run", check_every=10, precision="fp64",
               time_scheme="TVD_RK3", order="Second", limiter="Barth", flux="Rusanov", cell_order="morton",
               lts=False, check=False, cfl=0.5)
    return [
        # the reference's own calling pattern (Driver: calc_timestep, step, from the host) on
        # the smallest useful mesh: launches and host round trips are all there is
        dict(box, name="tet_host_steps_1k", n0=6, n1=6, n2=6, jitter=0.1, bc="SlipWall", mode="host", steps=10),
        # a plain steady solve of a channel with a bump (the steady benchmark's baseline, its
        # usual size): unlimited second order, CFL 1, residual looked at between graph replays
        dict(box, name="tet_channel_44k", mesh="channel", k=9, steps=100, check_every=50, limiter="NONE", cfl=1.0,
             drop=1e-8, jitter=0.0),
        # an ordinary transient run in a box, ragged sizes
        dict(box, name="tet_box_500k", n0=47, n1=45, n2=41, steps=40),
        # the headline step: 128^3 x 6 tetrahedra, upload, steps on the device, download
        dict(box, name="tet_box_12m", n0=128, n1=128, n2=128, steps=20),
        # the same step with FP32 face arithmetic
        dict(box, name="tet_box_mixed_1m", n0=61, n1=60, n2=59, steps=40, precision="mixed"),
        # several uneven channels in one batch, local time steps, mixed precision: how the
        # library's steady studies run (8 instances of 20k to 60k cells)
        dict(name="batch_channels_mixed", kind="batch", instances=8, k=7, k_spread=4, steps=100, check_every=50,
             precision="mixed", lts=True, limiter="NONE", cfl=1.0),
        # hexahedra: the mixed-element path
        dict(box, name="hex_box_500k", mesh="hex", n0=88, n1=79, n2=75, steps=20),
        # hexahedra and wedges stepped from the host on a small mesh with the physical-validity check,
        # as an input.yml of a small mixed mesh asks for
        dict(box, name="wedge_host_steps_2k", mesh="wedge", n0=13, n1=11, n2=12, bc="SlipWall", mode="host", steps=5,
             check=True, jitter=0.1),
        # every field a debug output writes: gradient, limiter, flux balance, primitive variables
        dict(box, name="fields_400k", kind="fields", n0=42, n1=40, n2=38),
        # learned warm start of a channel at the size the networks are used at: features,
        # inference, state
        dict(name="warm_start_1m", kind="warm", k=29),
        # inference for a serving loop: device arrays, a few hundred samples
        dict(name="mlp_predict_device_700", kind="predict_device", samples=700),
        # training the network: two epochs over a sampled solution set, minibatches of 2048
        dict(name="mlp_train_60k", kind="train", samples=60000, batch=2048, epochs=2),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "solve", "solve", "batch", "fields", "warm", "features", "predict",
                       "predict_device", "train", "loss_grad"])
    if kind in ("solve", "fields"):
        mesh = rng.choice(["tet", "tet", "tet", "hex", "wedge"]) if kind == "solve" else rng.choice(["tet", "hex"])
        lo, hi = (60, 1.5e6) if mesh == "tet" else (40, 4e5) if mesh == "hex" else (40, 3e4)
        if kind == "fields":
            hi = min(hi, 4e5)
        blocks = math.exp(rng.uniform(math.log(lo), math.log(hi))) / (6 if mesh == "tet" else 1)
        a, b = rng.uniform(0.7, 1.4), rng.uniform(0.7, 1.4)
        s = blocks ** (1 / 3)
        c = dict(kind=kind, mesh=mesh, n0=max(2, round(s * a)), n1=max(2, round(s * b)), n2=max(2, round(s / (a * b))),
                 bc=rng.choice(["FarField", "SlipWall"]), jitter=rng.choice([0.0, 0.1, 0.15]),
                 precision="mixed" if mesh == "tet" and rng.random() < 0.3 else "fp64",
                 time_scheme=rng.choice(["TVD_RK3", "TVD_RK3", "ExplicitEuler"]),
                 order=rng.choice(["Second", "Second", "Second", "First"]), limiter=rng.choice(["Barth", "Barth", "NONE"]),
                 cell_order=rng.choice(["morton", "morton", "rcm", "input"]), lts=rng.random() < 0.25,
                 check=rng.random() < 0.2, cfl=rng.choice([0.3, 0.5]))
        c["flux"] = "HLLC" if c["precision"] == "fp64" and rng.random() < 0.15 else "Rusanov"
        if kind == "fields":
            c["order"] = "Second"
        else:
            c.update(mode=rng.choice(["run", "run", "host"]), steps=rng.randint(3, 40), check_every=rng.choice([1, 5, 10]))
            if c["mode"] == "host":
                c["steps"] = min(c["steps"], 10)
        return c
    if kind == "batch":
        return dict(kind=kind, instances=rng.randint(2, 12), k=rng.randint(2, 8), k_spread=rng.randint(1, 4),
                    steps=rng.randint(10, 100), check_every=rng.choice([10, 25]), precision=rng.choice(["mixed", "fp64"]),
                    lts=rng.random() < 0.7, limiter=rng.choice(["NONE", "Barth"]), cfl=0.5)
    if kind in ("warm", "features"):
        return dict(kind=kind, k=_log_int(rng, 3, 27))
    if kind == "predict":
        return dict(kind=kind, samples=_log_int(rng, 1, 1.5e6))
    if kind == "predict_device":
        return dict(kind=kind, samples=_log_int(rng, 1, 16384))
    if kind == "train":
        return dict(kind=kind, samples=_log_int(rng, 2048, 120000), batch=256 * rng.randint(1, 16), epochs=rng.randint(1, 2))
    return dict(kind=kind, samples=_log_int(rng, 1, 2e5))


# ---------------------------------------------------------------------------
# meshes: nodes, cells and boundary faces as arrays
def _grid(n, lengths, jitter, bump):
    """Nodes of an n[0] x n[1] x n[2] block grid (x fastest), interior nodes
    moved by up to jitter x spacing; bump: height of a Gaussian floor bump."""
    n = np.array(n)
    I = np.stack(np.meshgrid(*[np.arange(m + 1) for m in n[::-1]], indexing="ij")[::-1], -1).reshape(-1, 3)
    h = np.array(lengths) / n
    X = I * h
    if jitter > 0:
        inner = ((I > 0) & (I < n)).all(1)
        X[inner] += (np.random.default_rng(20260101).random((int(inner.sum()), 3)) - 0.5) * (2 * jitter * h)
    if bump > 0:
        yb = bump * np.exp(-((X[:, 0] - 0.5 * lengths[0]) ** 2) / (2 * 0.2 ** 2))
        X[:, 1] = yb + X[:, 1] * (1 - yb / lengths[1])
    return X


def _sides(n, idx):
    """The four corners of every block face of the six sides x-, x+, ... z+,
    as (lower, first axis, both, second axis) node ids."""
    for ax in range(3):
        a, b = [d for d in range(3) if d != ax]
        u, v = [w.ravel() for w in np.meshgrid(np.arange(n[a]), np.arange(n[b]), indexing="ij")]
        for end in (0, n[ax]):
            q = [None] * 3

            def at(du, dv):
                q[ax], q[a], q[b] = np.full_like(u, end), u + du, v + dv
                return idx(*q)
            yield ax, np.stack([at(0, 0), at(1, 0), at(1, 1), at(0, 1)], 1)


@functools.lru_cache(maxsize=4)
def mesh_arrays(mesh, n, lengths, jitter, bump):
    """(nodes, [(element name, cells)], per side [(triangles or quads)])"""
    X = _grid(n, lengths, jitter, bump)
    i, j, k = [w.ravel() for w in np.meshgrid(*[np.arange(m) for m in n[::-1]], indexing="ij")[::-1]]

    def idx(i, j, k):
        return (i + (n[0] + 1) * (j + (n[1] + 1) * k)).astype(np.uint32)

    sides = [[] for _ in range(6)]
    if mesh == "tet":  # six tetrahedra per block around its (0,0,0)-(1,1,1) diagonal
        cells = []
        for p in ((0, 1, 2), (0, 2, 1), (1, 0, 2), (1, 2, 0), (2, 0, 1), (2, 1, 0)):
            d, v = [0, 0, 0], [idx(i, j, k)]
            for ax in p:
                d[ax] = 1
                v.append(idx(i + d[0], j + d[1], k + d[2]))
            if p in ((0, 2, 1), (1, 0, 2), (2, 1, 0)):
                v[1], v[2] = v[2], v[1]
            cells.append(np.stack(v, 1))
        cells = np.stack(cells, 1).reshape(-1, 4)
        for s, (_, q) in enumerate(_sides(n, idx)):
            sides[s].append(np.concatenate([q[:, [0, 1, 2]], q[:, [0, 2, 3]]]))
        return X, [("tet", cells)], sides
    v = np.stack([idx(i, j, k), idx(i + 1, j, k), idx(i + 1, j + 1, k), idx(i, j + 1, k),
                  idx(i, j, k + 1), idx(i + 1, j, k + 1), idx(i + 1, j + 1, k + 1), idx(i, j + 1, k + 1)], 1)
    split = (i + 2 * j) % 3 == 1 if mesh == "wedge" else np.zeros(len(i), bool)
    groups = [("hex", v[~split])]
    if split.any():  # two wedges per block, split through its (x, y) diagonal
        w = v[split]
        groups.append(("wedge", np.concatenate([w[:, [0, 2, 1, 4, 6, 5]], w[:, [0, 3, 2, 4, 7, 6]]])))
    for s, (ax, q) in enumerate(_sides(n, idx)):
        if ax == 2 and split.any():
            a, b = np.meshgrid(np.arange(n[0]), np.arange(n[1]), indexing="ij")
            sp = ((a + 2 * b) % 3 == 1).ravel()
            sides[s] += [q[~sp], q[sp][:, [0, 1, 2]], q[sp][:, [0, 2, 3]]]
        else:
            sides[s].append(q)
    return X, groups, sides


def mesh_key(c, h=None, k=None):
    if c.get("mesh", "channel") == "channel":
        k = c["k"] if k is None else k
        return "tet", (5 * k, 2 * k, k), (3.0, 1.0, 0.5), 0.0, 0.05 if h is None else h
    return c["mesh"], (c["n0"], c["n1"], c["n2"]), (1.0, 1.0, 1.0), c["jitter"], 0.0


def boundary(c):
    return ("FarField", "FarField") + ("SlipWall",) * 4 if c.get("mesh", "channel") == "channel" else (c["bc"],) * 6


@functools.lru_cache(maxsize=12)
def _mesh(key, bcs):
    X, groups, sides = mesh_arrays(*key)
    if key[0] == "tet":
        return nf.Mesh.from_arrays(X, groups[0][1], [s[0] for s in sides], bcs)
    if len(groups) == 1:
        return nf.Mesh.from_elements(X, groups[0][1], [s[0] for s in sides], bcs)
    rows = [list(r) for _, g in groups for r in g]
    return nf.Mesh.from_elements(X, rows, [[list(r) for q in s for r in q] for s in sides], bcs)


# ---------------------------------------------------------------------------
# states
def _config(c, mach):
    return nf.Config(time_scheme=c.get("time_scheme", "TVD_RK3"), spatial_order=c.get("order", "Second"),
                     limiter=c["limiter"], inviscid_flux_scheme=c.get("flux", "Rusanov"), CFL=c["cfl"], density_fs=1.0,
                     velocity_fs=(mach, 0.0, 0.0), pressure_fs=1 / GAMMA, check_physical_validity=c.get("check", False),
                     rk3_zero_old_first_step=False, precision=c["precision"], cell_order=c.get("cell_order", "morton"),
                     local_time_step=c["lts"])


def _mach(seed):
    return 0.3 + 0.4 * ((seed * 2654435761) % 1000003) / 1000003


@functools.lru_cache(maxsize=4)
def _centres(key):
    X, groups, _ = mesh_arrays(*key)
    return np.concatenate([X[g].mean(1) for _, g in groups])


def _cons(V):
    U = np.empty_like(V)
    U[:, 0] = V[:, 0]
    U[:, 1:4] = V[:, :1] * V[:, 1:4]
    U[:, 4] = V[:, 4] / (GAMMA - 1) + 0.5 * V[:, 0] * (V[:, 1:4] ** 2).sum(1)
    return U


def _state(c, key, seed, mach):
    """A freestream with a density pulse in a box (its place and height from
    the seed), the freestream itself in a channel."""
    x = _centres(key)
    V = np.zeros((len(x), 5))
    V[:, 0], V[:, 1], V[:, 4] = 1.0, mach, 1 / GAMMA
    if c.get("mesh", "channel") != "channel":
        if c["bc"] == "SlipWall":
            V[:, 1] = 0.0
        r = np.random.default_rng(seed)
        centre, amp = r.uniform(0.3, 0.7, 3), r.uniform(0.05, 0.15)
        V[:, 0] += amp * np.exp(-((x - centre) ** 2).sum(1) / (2 * 0.1 ** 2))
        V[:, 4] *= V[:, 0] ** GAMMA
    return _cons(V)


# ---------------------------------------------------------------------------
def _features_like(n, seed):
    """Samples as the features of channel cells are distributed."""
    r = np.random.default_rng(seed)
    x = r.random((n, 6)) * np.array([0.5, 0.08, 3.0, 1.0, 0.5, 0.25]) + np.array([0.3, 0.02, 0, 0, 0, 0])
    return x.astype(np.float32)


def _flow_like(x, seed):
    """Smooth primitive variables over such samples, and a little noise."""
    r = np.random.default_rng(seed + 1)
    b = x[:, 1] * np.exp(-((x[:, 2] - 1.5) ** 2) / 0.08) * np.exp(-3 * x[:, 3])
    y = np.stack([1 - 0.5 * x[:, 0] * b, x[:, 0] * (1 + 2 * b), -x[:, 0] * b * (x[:, 2] - 1.5) * 4, 0 * b,
                  1 / GAMMA - x[:, 0] ** 2 * b], 1)
    return (y + 1e-3 * r.standard_normal(y.shape)).astype(np.float32)


def _batch_dims(c):
    return [(c["k"] + q % c["k_spread"], 0.02 + 0.01 * (q % 8)) for q in range(c["instances"])]


def prepare(case, seed):
    c, s = case, dict(case=case)
    kind = c["kind"]
    if kind in ("solve", "fields"):
        key, mach = mesh_key(c), _mach(seed)
        s["cfg"] = _config(c, mach)
        s["U0"] = _state(c, key, seed, mach)
        s["solver"] = nf.EulerSolver(s["cfg"], _mesh(key, boundary(c)))
        if kind == "fields":
            s["solver"].set_state(s["U0"])
    elif kind == "batch":
        s["mach"] = [_mach(seed + 17 * q) for q in range(c["instances"])]
        keys = [mesh_key(c, h, k) for k, h in _batch_dims(c)]
        s["U0"] = [_state(c, key, seed, m) for key, m in zip(keys, s["mach"])]
        s["batch"] = nf.BatchSolver([_config(c, m) for m in s["mach"]], [_mesh(key, boundary(c)) for key in keys])
    elif kind in ("warm", "features"):
        s["params"] = (_mach(seed), 0.05)
        cfg = _config(dict(limiter="NONE", cfl=1.0, precision="fp64", lts=True), s["params"][0])
        s["batch"] = nf.BatchSolver([cfg], [_mesh(mesh_key(c), boundary(c))])
        s["net"], _ = _network()
    elif kind in ("predict", "predict_device"):
        s["net"], _ = _network()
        s["x"] = _features_like(c["samples"], seed)
        if kind == "predict_device":
            s["x"] = torch.from_numpy(s["x"]).cuda()
            s["y"] = torch.zeros(c["samples"], 5, device="cuda")
            s["stream"] = torch.cuda.Stream()
            torch.cuda.synchronize()
    else:
        s["net"] = Mlp(seed % 1000)
        s["p0"] = s["net"].params
        s["x"] = _features_like(c["samples"], seed)
        s["y"] = _flow_like(s["x"], seed)
        s["net"].set_norm(*_norm_of(s["x"], s["y"]))
    return s


def _network():
    return steady.load_network(os.path.join(ROOT, NETWORK))


def _norm_of(x, y):
    return (x.mean(0), 1 / np.maximum(x.std(0), 1e-3), y.mean(0), np.maximum(y.std(0), 0.01))


# ---------------------------------------------------------------------------
def run(state):
    return globals()["run_" + state["case"]["kind"]](state)


def run_solve(s):
    """Initial state in, time steps, state and residual history out."""
    c, solver, cfg = s["case"], s["solver"], s["cfg"]
    solver.set_state(s["U0"], s["U0"])
    out = {}
    if c["mode"] == "host":
        dt = []
        for _ in range(c["steps"]):
            solver.calc_timestep(cfg)
            solver.step(cfg)
            dt.append(cfg.delta_time)
        out["dt"] = np.array(dt)
    else:
        out["time"] = solver.run(c["steps"], residual_drop=c.get("drop", 0.0), check_every=c["check_every"])["time"]
    out["U"] = solver.get_solver_data().get_solution()
    out["residuals"] = solver.residuals(max_n=1024)
    return out


def run_fields(s):
    """What a debug output writes, for a state in hand."""
    solver = s["solver"]
    data = solver.get_solver_data()
    solver.eval_flux_balance()
    return {"grad": data.get_primvars_gradient(), "psi": data.get_primvars_limiter(), "R": data.get_flux_balance(),
            "V": data.get_primvars()}


def run_batch(s):
    """A batched steady solve's start: freestream states, their residuals as
    the references of the drop, steps, solutions."""
    c, b = s["case"], s["batch"]
    for q, U in enumerate(s["U0"]):
        b.set_state(q, U, U)
    ref = b.eval_residuals()
    for q, r in enumerate(ref):
        b.set_residual_ref(q, r)
    b.run(c["steps"], residual_drop=1e-8, check_every=c["check_every"])
    return {"ref": ref, "U": [b.get_solution(q) for q in range(b.n)], "res": [b.residuals(q, 1024) for q in range(b.n)]}


def run_warm(s):
    fell = s["batch"].warm_start(0, s["net"], s["params"])
    return {"fell_back": int(fell), "U": s["batch"].get_solution(0)}


def run_features(s):
    return s["batch"].features(0, s["params"])


def run_predict(s):
    return s["net"].predict(s["x"])


def run_predict_device(s):
    rc = _abi.lib().nf_mlp_predict_noalloc(s["net"]._h, s["x"].data_ptr(), s["case"]["samples"], s["y"].data_ptr(),
                                           s["stream"].cuda_stream)
    if rc:
        raise RuntimeError("nf_mlp_predict_noalloc: status %d" % rc)
    return s["y"]


def run_train(s):
    c, net = s["case"], s["net"]
    net.params = s["p0"]
    st = net.train(s["x"], s["y"], epochs=c["epochs"], batch=c["batch"], lr=2e-3, lr_decay=0.98, seed=7)
    return {"params": net.params, "loss_first": st["loss_first"], "loss_last": st["loss_last"]}


def run_loss_grad(s):
    loss, grad = s["net"].loss_grad(s["x"], s["y"])
    return {"loss": loss, "grad": grad}


# ---------------------------------------------------------------------------
MLP_FLOPS = 2 * (6 * 128 + 2 * 128 * 128 + 128 * 5)


def n_cells(c):
    if c.get("mesh", "channel") == "channel":
        return 60 * c["k"] ** 3
    n = c["n0"] * c["n1"] * c["n2"]
    return 6 * n if c["mesh"] == "tet" else int(n * 4 / 3) if c["mesh"] == "wedge" else n


def work(case):
    """One pass: each stage reads the state, U_old (after the first) and the
    connectivity or slot geometry once and writes the state; arrays of the
    call itself once.  About 1500 (tetrahedra) or 2200 (hexahedra) floating
    point operations per cell and stage."""
    c, kind = case, case["kind"]
    if kind in ("solve", "batch", "fields"):
        N = n_cells(c) if kind != "batch" else sum(60 * k ** 3 for k, _ in _batch_dims(c))
        stages = 1 if kind == "fields" else c["steps"] * (3 if c.get("time_scheme", "TVD_RK3") == "TVD_RK3" else 1)
        tet = c.get("mesh", "channel") in ("tet", "channel")
        per_stage = 40 + 40 + (27 if stages > 1 else 0) + (40 if tet else 180)
        ends = 240 if kind == "fields" else 80
        return {"bytes": N * (stages * per_stage + ends), "flops": N * stages * (1500 if tet else 2200)}
    if kind in ("warm", "features"):
        N = 60 * c["k"] ** 3
        return {"bytes": N * (56 + (80 if kind == "warm" else 24)), "flops": N * (100 + (MLP_FLOPS if kind == "warm" else 0))}
    n = c["samples"]
    if kind == "train":
        seen = n // min(c["batch"], n // 256 * 256) * min(c["batch"], n // 256 * 256) * c["epochs"]
        return {"bytes": 44 * n + 44 * seen, "flops": 3 * MLP_FLOPS * seen}
    return {"bytes": 44 * n, "flops": (3 if kind == "loss_grad" else 1) * MLP_FLOPS * n}


# ---------------------------------------------------------------------------
# the same in plain torch FP64
def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _cross(a, b):
    return torch.linalg.cross(a, b, dim=-1)


def _tri(p):
    return 0.5 * _cross(p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]), p.sum(1) / 3


def _quad(p):
    (Sa, ca), (Sb, cb) = _tri(p[:, [0, 1, 2]]), _tri(p[:, [0, 2, 3]])
    a, b = Sa.norm(dim=1, keepdim=True), Sb.norm(dim=1, keepdim=True)
    return Sa + Sb, (a * ca + b * cb) / (a + b)


def _cell_geometry(name, p):
    """Volumes and centroids: a tetrahedron's own; hexahedra and wedges as
    the pyramids and tetrahedra over their faces around the node mean."""
    if name == "tet":
        d = p[:, 1:] - p[:, :1]
        return (_cross(d[:, 0], d[:, 1]) * d[:, 2]).sum(1).abs() / 6, p.mean(1)
    g = p.mean(1)
    vol, mom = 0, 0
    for f in PARTS[name]:
        S, c = (_quad if len(f) == 4 else _tri)(p[:, list(f)])
        v = ((c - g) * S).sum(1, keepdim=True).abs() / 3
        vol, mom = vol + v, mom + v * (0.75 * c + 0.25 * g)
    return vol[:, 0], mom / vol


FACES = {"tet": ((0, 1, 2), (0, 1, 3), (0, 2, 3), (1, 2, 3)),
         "hex": ((0, 1, 2, 3), (4, 5, 6, 7), (0, 1, 5, 4), (3, 2, 6, 7), (3, 0, 4, 7), (1, 2, 6, 5)),
         "wedge": ((0, 1, 2), (4, 3, 5), (1, 0, 3, 4), (0, 2, 5, 3), (4, 5, 2, 1))}
# bases of the pyramids and tetrahedra of a cell's volume; where a quadrilateral
# is not plane, its centroid depends on the diagonal (first to third node)
PARTS = {"hex": ((0, 1, 2, 3), (4, 7, 6, 5), (4, 0, 3, 7), (2, 1, 5, 6), (1, 0, 4, 5), (3, 2, 6, 7)),
         "wedge": ((0, 2, 1), (3, 4, 5), (0, 3, 5, 2), (0, 1, 4, 3), (4, 1, 2, 5))}


class Reference:
    """Face graph, geometry and one flux evaluation in torch FP64."""

    def __init__(self, key, bcs, Vinf):
        X, groups, sides = mesh_arrays(*key)
        dev = _dev()
        X = torch.from_numpy(X).to(dev)
        vol, cen, key_, own, nodes, first = [], [], [], [], [], 0
        for name, g in groups:
            g = torch.from_numpy(g.astype(np.int64)).to(dev)
            v, m = _cell_geometry(name, X[g])
            vol.append(v)
            cen.append(m)
            for f in FACES[name]:
                q = g[:, list(f)]
                if q.shape[1] == 3:
                    q = torch.cat([q, torch.full_like(q[:, :1], -1)], 1)
                nodes.append(q)
                own.append(torch.arange(first, first + len(g), device=dev))
            first += len(g)
        self.N, self.vol, self.cen = first, torch.cat(vol), torch.cat(cen)
        nodes, own = torch.cat(nodes), torch.cat(own)
        key_ = self._key(nodes, len(X))
        key_, at = torch.sort(key_, stable=True)
        pair = torch.zeros(len(at), dtype=torch.bool, device=dev)
        pair[:-1] = key_[1:] == key_[:-1]
        second = torch.zeros_like(pair)
        second[1:] = pair[:-1]
        a, b = at[pair], at[torch.roll(pair, 1, 0)]
        alone = ~(pair | second)
        lone, lone_key = at[alone], key_[alone]
        a, b = torch.where(own[a] < own[b], a, b), torch.where(own[a] < own[b], b, a)
        fi, fj, fn = own[a], own[b], nodes[a]  # the lower cell's node order is the face's
        bc = torch.full((len(lone),), -1, device=dev)
        for s, q in enumerate(sides):
            for w in q:
                w = torch.from_numpy(w.astype(np.int64)).to(dev)
                if w.shape[1] == 3:
                    w = torch.cat([w, torch.full_like(w[:, :1], -1)], 1)
                bc[torch.searchsorted(lone_key, self._key(w, len(X)))] = 1 if bcs[s] == "FarField" else 0
        self.F, self.far = len(fi), bc == 1
        self.i, self.j = torch.cat([fi, own[lone]]), fj
        fn = torch.cat([fn, nodes[lone]])
        S, c = torch.empty(len(fn), 3, dtype=X.dtype, device=dev), torch.empty(len(fn), 3, dtype=X.dtype, device=dev)
        t = fn[:, 3] < 0
        S[t], c[t] = _tri(X[fn[t][:, :3]])
        S[~t], c[~t] = _quad(X[fn[~t]])
        out = ((c - self.cen[self.i]) * S).sum(1, keepdim=True) < 0
        self.S = torch.where(out, -S, S)
        self.ri, self.rj = c - self.cen[self.i], c[:self.F] - self.cen[self.j]
        self.dS = torch.zeros(self.N, 3, dtype=X.dtype, device=dev)
        self.dS.index_add_(0, fi, 0.5 * self.S[:self.F].abs())
        self.dS.index_add_(0, fj, 0.5 * self.S[:self.F].abs())
        self.wall_c = c[self.F:][~self.far]
        self.Vinf = torch.tensor(Vinf, dtype=torch.float64, device=dev)

    @staticmethod
    def _key(nodes, n):
        """One number per face from its three largest nodes, which no two
        faces of these meshes share (products may wrap around; at up to 2.6
        million nodes they still differ)."""
        q = torch.sort(nodes, 1).values
        return (q[:, 1] * n + q[:, 2]) * n + q[:, 3]

    @staticmethod
    def prim(U):
        V = torch.empty_like(U)
        V[:, 0] = U[:, 0]
        V[:, 1:4] = U[:, 1:4] / U[:, :1]
        V[:, 4] = (GAMMA - 1) * (U[:, 4] - 0.5 * (U[:, 1:4] ** 2).sum(1) / U[:, 0])
        return V

    def ghost(self, V):
        """Boundary states of the faces' inner states: slip wall, or farfield
        from the Riemann invariants."""
        S = self.S[self.F:]
        n = S / S.norm(dim=1, keepdim=True)
        vn = (V[:, 1:4] * n).sum(1, keepdim=True)
        G = V.clone()
        G[:, 1:4] -= 2 * vn * n
        if self.far.any():
            f, g1 = self.Vinf, GAMMA - 1
            nf_, vd = n[self.far], V[self.far]
            vnf, vnd = (nf_ * f[1:4]).sum(1), vn[self.far][:, 0]
            cf, cd = torch.sqrt(GAMMA * f[4] / f[0]), torch.sqrt(GAMMA * vd[:, 4] / vd[:, 0])
            Rp = torch.where(vnf + cf > 0, vnd + 2 * cd / g1, vnf + 2 * cf / g1)
            Rm = torch.where(vnf - cf > 0, vnd - 2 * cd / g1, vnf - 2 * cf / g1)
            vb, cb = 0.5 * (Rp + Rm), g1 / 4 * (Rp - Rm)
            out = (vnf > 0)[:, None]
            vel = torch.where(out, vd[:, 1:4] + (vb - vnd)[:, None] * nf_, f[1:4] + (vnf - vb)[:, None] * nf_)
            s = torch.where(vnf > 0, vd[:, 4] * vd[:, 0] ** -GAMMA, f[4] * f[0] ** -GAMMA)
            rho = (GAMMA * s / cb ** 2) ** (1 / g1)
            G[self.far] = torch.cat([rho[:, None], vel, (cb ** 2 * rho / GAMMA)[:, None]], 1)
        return G

    def cell_dt(self, V, cfl):
        c = torch.sqrt(GAMMA * V[:, 4] / V[:, 0])[:, None]
        return cfl * self.vol / ((V[:, 1:4].abs() + c) * self.dS).sum(1)

    def balance(self, V, second, barth):
        """(R, gradient, limiter) of the primitive variables V."""
        F, i, j = self.F, self.i, self.j
        Vi = V[i]
        Vj = torch.cat([V[j], self.ghost(Vi[F:])])
        grad = torch.zeros(self.N, 5, 3, dtype=V.dtype, device=V.device)
        psi = torch.ones_like(V)
        if second:
            t = (0.5 * (Vi + Vj))[:, :, None] * self.S[:, None, :]
            grad.index_add_(0, i, t)
            grad.index_add_(0, j, -t[:F])
            del t
            grad /= self.vol[:, None, None]
            di = (grad[i] * self.ri[:, None, :]).sum(2)
            dj = (grad[j] * self.rj[:, None, :]).sum(2)
            if barth:
                hi, lo = V.clone(), V.clone()
                at = i[:, None].expand(-1, 5)
                hi.scatter_reduce_(0, at, Vj, "amax")
                lo.scatter_reduce_(0, at, Vj, "amin")
                at = j[:, None].expand(-1, 5)
                hi.scatter_reduce_(0, at, Vi[:F], "amax")
                lo.scatter_reduce_(0, at, Vi[:F], "amin")
                for c, d in ((i, di), (j, dj)):
                    up, down = hi[c] - V[c], lo[c] - V[c]
                    eps = np.finfo(np.float64).eps
                    p = torch.where(d > 0, up / (d + eps), torch.where(d < 0, down / (d - eps), torch.ones_like(d)))
                    psi.scatter_reduce_(0, c[:, None].expand(-1, 5), p.clamp(max=1.0), "amin")
            Vi = Vi + psi[i] * di
            Vj = torch.cat([V[j] + psi[j] * dj, self.ghost(Vi[F:])])
        area = self.S.norm(dim=1, keepdim=True)
        n = self.S / area

        def flux(W):
            vn = (W[:, 1:4] * n).sum(1, keepdim=True)
            E = W[:, 4:] / (GAMMA - 1) + 0.5 * W[:, :1] * (W[:, 1:4] ** 2).sum(1, keepdim=True)
            U = torch.cat([W[:, :1], W[:, :1] * W[:, 1:4], E], 1)
            f = vn * U
            f[:, 1:4] += W[:, 4:] * n
            f[:, 4:] += vn * W[:, 4:]
            return U, f, vn.abs() + torch.sqrt(GAMMA * W[:, 4:] / W[:, :1])
        Ui, fi, si = flux(Vi)
        Uj, fj, sj = flux(Vj)
        f = 0.5 * area * (fi + fj - torch.maximum(si, sj) * (Uj - Ui))
        R = torch.zeros_like(V)
        R.index_add_(0, i, -f)
        R.index_add_(0, j, f[:F])
        return R, grad, psi

    def solve(self, U, c, steps):
        rk3 = c.get("time_scheme", "TVD_RK3") == "TVD_RK3"
        second, barth = c.get("order", "Second") == "Second", c["limiter"] == "Barth"
        U = torch.from_numpy(U).to(self.S.device)
        V, dts, res = self.prim(U), [], []
        for _ in range(steps):
            dt = self.cell_dt(V, c["cfl"]).min()  # of the primitive variables the last stage read
            dts.append(dt.item())
            V = self.prim(U)
            h = ((self.cell_dt(V, c["cfl"]) if c["lts"] else dt) / self.vol)[..., None]
            R = self.balance(V, second, barth)[0]
            res.append(R[:, 0].norm().item())
            old, U = U, U + h * R
            if rk3:
                U = 0.75 * old + 0.25 * U + 0.25 * h * self.balance(self.prim(U), second, barth)[0]
                V = self.prim(U)
                U = old / 3 + 2 / 3 * U + 2 / 3 * h * self.balance(V, second, barth)[0]
        return U.cpu().numpy(), np.array(dts), np.array(res)


def _forward(p, norm, x):
    """The network in FP64: x [n][6] raw -> normalised outputs [n][5]."""
    W = [p[s].reshape(shape) for s, shape in param_slices()]
    a = (x - norm[0]) * norm[1]
    for q in range(3):
        a = torch.nn.functional.gelu(a @ W[2 * q].T + W[2 * q + 1])
    return a @ W[6].T + W[7]


def _exact_predict(x):
    with np.load(os.path.join(ROOT, NETWORK), allow_pickle=False) as z:
        p = torch.from_numpy(z["params"].astype(np.float64)).to(_dev())
        norm = [torch.from_numpy(z[k].astype(np.float64)).to(_dev()) for k in ("in_shift", "in_scale", "out_shift", "out_scale")]
    y = torch.cat([_forward(p, norm, q) for q in x.double().to(_dev()).split(1 << 18)])
    return y * norm[3] + norm[2]


def _exact_features(c, seed):
    r = Reference(mesh_key(c), boundary(c), [1.0, _mach(seed), 0, 0, 1 / GAMMA])
    d = []
    for q in r.cen.split(max(1, (1 << 27) // max(1, len(r.wall_c)))):
        d2 = 0
        for ax in range(3):
            d2 = d2 + (q[:, ax:ax + 1] - r.wall_c[None, :, ax]) ** 2
        d.append(d2.min(1).values.sqrt())
    one = torch.ones_like(r.vol)[:, None]
    return torch.cat([one * _mach(seed), one * 0.05, r.cen, torch.cat(d)[:, None]], 1)


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("solve", "fields"):
        if c["flux"] != "Rusanov":
            return None
        key, mach = mesh_key(c), _mach(seed)
        r = Reference(key, boundary(c), [1.0, mach, 0.0, 0.0, 1 / GAMMA])
        U0 = _state(c, key, seed, mach)
        if kind == "fields":
            V = r.prim(torch.from_numpy(U0).to(_dev()))
            R, grad, psi = r.balance(V, c["order"] == "Second", c["limiter"] == "Barth")
            # the limiter of a constant region is 0 or 1 by rounding alone: no value for it
            return {"grad": grad.permute(0, 2, 1).reshape(-1, 15).cpu().numpy(), "psi": None, "R": R.cpu().numpy(),
                    "V": V.cpu().numpy()}
        U, dt, res = r.solve(U0, c, c["steps"])
        # (with local steps the global one is reported, but not used)
        t = {"dt": dt} if c["mode"] == "host" else {"time": float(dt.sum())}
        return {**{k: None if c["lts"] else v for k, v in t.items()}, "U": U, "residuals": res}
    if kind == "batch":
        ref, Us, rs = [], [], []
        for q, (k, h) in enumerate(_batch_dims(c)):
            key, mach = mesh_key(c, h, k), _mach(seed + 17 * q)
            r = Reference(key, boundary(c), [1.0, mach, 0.0, 0.0, 1 / GAMMA])
            U, _, res = r.solve(_state(c, key, seed, mach), c, c["steps"])
            ref.append(res[0])
            Us.append(U)
            rs.append(res)
        return {"ref": np.array(ref), "U": Us, "res": rs}
    if kind == "features":
        return _exact_features(c, seed).cpu().numpy()
    if kind == "warm":
        V = _exact_predict(_exact_features(c, seed))
        return {"fell_back": 0, "U": _cons(V.cpu().numpy())}
    if kind in ("predict", "predict_device"):
        return _exact_predict(torch.from_numpy(_features_like(c["samples"], seed))).cpu().numpy()
    if kind == "loss_grad":
        x = _features_like(c["samples"], seed)
        y = _flow_like(x, seed)
        norm = [torch.from_numpy(np.asarray(v, np.float32).astype(np.float64)).to(_dev()) for v in _norm_of(x, y)]
        p = torch.from_numpy(Mlp(seed % 1000).params.astype(np.float64)).to(_dev()).requires_grad_()
        out = _forward(p, norm, torch.from_numpy(x).double().to(_dev()))
        loss = ((out - (torch.from_numpy(y).double().to(_dev()) - norm[2]) / norm[3]) ** 2).mean()
        loss.backward()
        return {"loss": loss.item(), "grad": p.grad.cpu().numpy()}
    return None  # training: hundreds of updates, each through 16-bit weights
