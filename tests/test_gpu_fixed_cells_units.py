"""Fixed-point cells of grids whose cells are many units (millimetre maps) and of
maps of any whole number of cells: points around cell faces, weights bit for bit
against the oracle.  Which of them take the fixed-point form is asserted on the
CPU (test_fixed_cells.py)."""
import numpy as np
import pytest

import oracle
from test_gpu_fixed_cells import _near_faces

pytestmark = pytest.mark.gpu
F32 = np.float32

# cells, units per cell, min
GRIDS = {
    "9 units": ((2000, 60, 20), 9.0, (0.0, -4.0, 1.0)),
    "40 units": ((600, 50, 20), 40.0, (0.0, -700.0, 11.0)),
    "250 units": ((200, 90, 20), 250.0, (1.0, -3.0, 0.0)),
    "1,000 units, not fixed": ((4000, 9, 8), 1000.0, (0.0, 0.0, 0.0)),
    "19.9 m": ((199, 199, 60), 0.1, (0.0, 0.0, 0.0)),
    "4,000 cells": ((4000, 9, 8), 0.05, (-100.0, 0.0, 0.0)),
    "0.2 m": ((90, 300, 33), 0.2, (-9.0, 1e-3, 5.0)),
    "0.3 m": ((100, 77, 25), 0.3, (2.7, -11.0, -3.0)),
}


@pytest.mark.parametrize("name", list(GRIDS))
@pytest.mark.parametrize("poses", [3, 2500, 29000])
def test_points_near_cell_faces(gpu, name, poses):
    n, res, mn = GRIDS[name]
    n, mn = np.array(n), np.array(mn)
    mx = mn + n * res
    n = np.ceil((mx - mn) / res).astype(int)
    prob = np.random.default_rng(len(name)).uniform(0.0, 4.0, (n[2], n[1], n[0])).astype(F32)
    g, og = gpu.Grid3d().from_cells(prob, mn, mx, res, 0.1), oracle.GridMeta(mn, mx, res, prob)
    rng = np.random.default_rng(poses)
    pose = (mn + (mx - mn) * rng.uniform(0.1, 0.9, 3)).astype(F32)
    cloud = _near_faces(rng, pose, mn, res, n, 3000 if poses < 100 else 200)
    t = np.tile(np.append(pose, F32(0)), (poses, 1)).astype(F32)
    t[1::3, :3] += (rng.integers(-3, 4, (len(t[1::3]), 3)) * res).astype(F32)
    t[2::3, :3] = mn + (mx - mn) * rng.uniform(-0.05, 1.05, (len(t[2::3]), 3))
    t[2::3, 3] = rng.uniform(-3.2, 3.2, len(t[2::3]))
    if poses > 100:
        far = np.array([2.0 ** 19, 2.0 ** 21, -2.0 ** 30, 2.0 ** 36]) * res  # cells past 2^20 away
        t[20:24, 0] = far
        cloud[:16, 0] = (-far[:, None] + mn[0] + rng.integers(0, n[0], 4) * res).ravel()
    for roll, pitch in ((0.0, 0.0), (0.03, -0.07)):
        w = g.cloud_weights(cloud, t[:, 0], t[:, 1], t[:, 2], t[:, 3], roll, pitch)
        ow = oracle.cloud_weight_batch(og, cloud, t[:, 0], t[:, 1], t[:, 2], t[:, 3], roll, pitch)
        assert np.array_equal(w.view(np.int32), ow.view(np.int32)), (name, roll)


@pytest.mark.parametrize("poses", [40, 2500, 7000, 29000])
def test_many_points_and_rotations_that_are_not_finite(gpu, poses):
    n, res, mn = GRIDS["19.9 m"]
    n, mn = np.array(n), np.array(mn)
    mx = mn + n * res
    prob = np.random.default_rng(7).uniform(0.0, 4.0, (n[2], n[1], n[0])).astype(F32)
    g, og = gpu.Grid3d().from_cells(prob, mn, mx, res, 0.1), oracle.GridMeta(mn, mx, res, prob)
    rng = np.random.default_rng(poses)
    cloud = rng.uniform(-5, 5, (300, 3)).astype(F32)
    bad = rng.random(300) < 0.4
    cloud[bad, rng.integers(0, 3, bad.sum())] = rng.choice([np.nan, np.inf, -np.inf], bad.sum())
    t = np.empty((poses, 4), F32)
    t[:, :3] = rng.uniform(mn, mx, (poses, 3))
    t[:, 3] = rng.uniform(-3.2, 3.2, poses)
    t[::2, :3] = np.round(t[::2, :3], 1)  # offsets on faces
    t[3::50, 3] = rng.choice([np.nan, np.inf], len(t[3::50]))
    for roll, pitch in ((0.0, 0.0), (0.03, -0.07), (np.nan, 0.0)):
        w = g.cloud_weights(cloud, t[:, 0], t[:, 1], t[:, 2], t[:, 3], roll, pitch)
        ow = oracle.cloud_weight_batch(og, cloud, t[:, 0], t[:, 1], t[:, 2], t[:, 3], roll, pitch)
        assert np.array_equal(w.view(np.int32), ow.view(np.int32)), roll
