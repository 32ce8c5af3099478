"""Network features against a brute-force scan of every wall-face centroid:
the pruned search on the device has to give the same minimum bit for bit, in
every cell numbering, with no wall, with fewer points than one box, with a
padded last box, and with walls on one side only."""
import numpy as np
import pytest

import netflux_amd as nf

pytestmark = pytest.mark.gpu

F, W = "FarField", "SlipWall"
CASES = {  # block counts, patches
    "no_wall": ((3, 3, 3), (F,) * 6),
    "one_block": ((1, 1, 1), ("NoSlipWall",) * 6),
    "one_side": ((5, 4, 3), (W,) + (F,) * 5),
    "box": ((13, 11, 9), (W,) * 6),
    "channel": ((30, 12, 6), (F, F) + (W,) * 4),
}


def _nearest(cen, wall):
    """min over the wall points of the FP32 distance, in the device's order of operations"""
    out = []
    for c in np.array_split(cen, max(1, len(cen) * len(wall) // 4_000_000)):
        d = [wall[None, :, k] - c[:, k:k + 1] for k in range(3)]
        out.append(np.sqrt(((d[0] * d[0] + d[1] * d[1]) + d[2] * d[2]).min(1)))
    return np.concatenate(out)


@pytest.mark.parametrize("order", ["morton", "rcm", "input"])
@pytest.mark.parametrize("name", list(CASES))
def test_features_match_a_full_scan(name, order):
    print(f"[case] features {name} {order}", flush=True)
    n, patches = CASES[name]
    mesh = nf.Mesh.box(n, lengths=(3.0, 1.0, 0.5), jitter=0.2, patches=patches)
    cfg = nf.Config(density_fs=1.0, velocity_fs=(0.5, 0, 0), pressure_fs=1 / 1.4, cell_order=order)
    x = nf.BatchSolver([cfg], [mesh]).features(0, (0.4, 0.06))
    nodes, cells, pn, pf, pbc = mesh.arrays()
    X = nodes[cells]
    cen = (0.25 * (((X[:, 0] + X[:, 1]) + X[:, 2]) + X[:, 3])).astype(np.float32)
    first = np.r_[0, np.cumsum(pn)]
    faces = [pf[first[q]:first[q + 1]] for q in range(len(pn)) if pbc[q] != 2]
    if faces:
        P = nodes[np.concatenate(faces)]
        dist = _nearest(cen, (((P[:, 0] + P[:, 1]) + P[:, 2]) / 3).astype(np.float32))
    else:
        dist = np.zeros(len(cen), np.float32)
    np.testing.assert_array_equal(x[:, :2], np.tile(np.array([0.4, 0.06], np.float32), (len(cen), 1)))
    np.testing.assert_array_equal(x[:, 2:5], cen)
    np.testing.assert_array_equal(x[:, 5], dist)
