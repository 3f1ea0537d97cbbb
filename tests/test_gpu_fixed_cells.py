"""The cloud weight's fixed-point cells (clean grids whose bounds are cell
faces): points on cell faces and a few float spacings either side of them, at
both ends of every axis, under poses of many offsets, and grids just outside
the rule; weights bit for bit against the oracle."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu
F32 = np.float32

# cells, metres per cell, min, how far max lies from the last face (cells)
GRIDS = {
    "0.1 m": ((200, 180, 60), 0.1, (0.0, 0.0, 0.0), 0.0),
    "0.05 m": ((900, 40, 70), 0.05, (-17.35, 3.1, -0.4), 0.0),
    "0.2 m": ((90, 300, 33), 0.2, (-9.0, 1e-3, 5.0), 0.0),
    "0.25 m": ((64, 128, 20), 0.25, (-8.0, -16.0, 0.0), 0.0),
    "0.3 m": ((100, 77, 25), 0.3, (2.7, -11.0, -3.0), 0.0),
    "7,000 cells": ((7000, 8, 9), 0.05, (-100.0, 0.0, 0.0), 0.0),
    "9,000 cells": ((9000, 8, 9), 0.05, (-100.0, 0.0, 0.0), 0.0),
    "half a last cell": ((120, 80, 30), 0.1, (0.0, 0.0, 0.0), 0.5),
    "a last cell of rounding": ((121, 81, 31), 0.1, (0.0, 0.0, 0.0), 1.0 - 1e-12),
    "not clean": ((150, 90, 40), 0.07, (0.0, -2.0, 0.0), 0.0),
}


def _grid(gpu, name):
    size, res, mn, cut = GRIDS[name]
    mn = np.array(mn)
    mx = mn + (np.array(size) - cut) * res
    n = np.ceil((mx - mn) / res).astype(int)
    prob = np.random.default_rng(len(name)).uniform(0.0, 4.0, (n[2], n[1], n[0])).astype(F32)
    return gpu.Grid3d().from_cells(prob, mn, mx, res, 0.1), oracle.GridMeta(mn, mx, res, prob), mn, mx, res, n


def _near_faces(rng, pose, mn, res, n, count):
    """Level points whose cells' faces lie within 3 float spacings on one to three axes (yaw 0: s is the point)."""
    c = np.empty((count, 3), F32)
    for a in range(3):
        k = rng.integers(-1, n[a] + 2, count)
        edge = rng.random(count) < 0.25
        k[edge] = rng.choice([0, n[a] - 1, n[a]], edge.sum())
        v = (k * res - (np.float64(pose[a]) - mn[a])).astype(F32)
        off = rng.random(count) < 0.35
        v[off] += rng.uniform(0, res, off.sum()).astype(F32)
        for _ in range(3):
            step = rng.integers(-1, 2, count)
            v = np.where(step > 0, np.nextafter(v, F32(np.inf)), np.where(step < 0, np.nextafter(v, F32(-np.inf)), v))
        c[:, a] = v
    return c


@pytest.mark.parametrize("name", list(GRIDS))
@pytest.mark.parametrize("poses", [3, 2500, 29000])
def test_points_near_cell_faces(gpu, name, poses):
    g, og, mn, mx, res, n = _grid(gpu, name)
    rng = np.random.default_rng(poses)
    pose = (mn + (mx - mn) * rng.uniform(0.1, 0.9, 3)).astype(F32)
    m = 3000 if poses < 100 else 200
    cloud = _near_faces(rng, pose, mn, res, n, m)
    t = np.tile(np.append(pose, F32(0)), (poses, 1)).astype(F32)
    # the same fractions of a cell at other cells, and other poses altogether
    t[1::3, :3] += (rng.integers(-3, 4, (len(t[1::3]), 3)) * res).astype(F32)
    t[2::3, :3] = mn + (mx - mn) * rng.uniform(-0.05, 1.05, (len(t[2::3]), 3))
    t[2::3, 3] = rng.uniform(-3.2, 3.2, len(t[2::3]))
    if poses > 100:
        t[5, :3] = mn  # zero offsets
        t[6, :3] = np.nextafter(mn.astype(F32), F32(np.inf))
        t[7, :3] = 1e9
        t[8, 0], t[11, 3] = np.inf, np.nan
    for roll, pitch in ((0.0, 0.0), (0.03, -0.07)):
        w = g.cloud_weights(cloud, t[:, 0], t[:, 1], t[:, 2], t[:, 3], roll, pitch)
        ow = oracle.cloud_weight_batch(og, cloud, t[:, 0], t[:, 1], t[:, 2], t[:, 3], roll, pitch)
        assert np.array_equal(w.view(np.int32), ow.view(np.int32)), (name, roll)


@pytest.mark.parametrize("poses", [40, 29000])
def test_extreme_points(gpu, poses):
    """Non-finite, huge, zero and subnormal points between ordinary ones."""
    g, og, mn, mx, res, n = _grid(gpu, "0.1 m")
    rng = np.random.default_rng(1)
    cloud = rng.uniform(-5, 5, (300, 3)).astype(F32)
    odd = [np.nan, np.inf, -np.inf, 3e38, -3e38, 1e30, 1e10, 0.0, -0.0, 1e-45, -1e-45, 1e-30]
    for k, v in enumerate(odd):
        cloud[7 * k, k % 3] = v
        cloud[7 * k + 100] = v
    t = np.tile(np.array([8.0, 9.0, 3.0, 0.0], F32), (poses, 1))
    t[1::2, 3] = rng.uniform(-3.1, 3.1, len(t[1::2]))
    t[3::4, :3] = mn
    w = g.cloud_weights(cloud, t[:, 0], t[:, 1], t[:, 2], t[:, 3])
    ow = oracle.cloud_weight_batch(og, cloud, t[:, 0], t[:, 1], t[:, 2], t[:, 3])
    assert np.array_equal(w.view(np.int32), ow.view(np.int32))
