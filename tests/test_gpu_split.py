"""The split form of the cloud weight (a workgroup's wavefronts share the cloud,
one more adds the values in order) at the sizes where its tiles, workgroups
and dispatch limits end: bit-exact against the oracle."""
import numpy as np
import pytest

import oracle
from amcl3d_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def room():
    c = W.room_case(1)
    bm = c["map"]
    pts = bm.points()
    _, prob = oracle.compute_grid(pts, bm.min, bm.max, bm.res, c["sensor_dev"], exp_mode=1)
    c.update(points=pts, ogrid=oracle.GridMeta(bm.min, bm.max, bm.res, prob))
    return c


def _open(gpu, room):
    g = gpu.Grid3d()
    bm = room["map"]
    g.open(room["points"], bm.min, bm.max, bm.res, room["sensor_dev"])
    return g


def _poses(room, n, seed=5):
    rng = np.random.default_rng(seed)
    base = room["particles"][rng.integers(0, len(room["particles"]), n)]
    t = base[:, :4] + rng.normal(0, 0.2, (n, 4)).astype(np.float32)
    if n > 8:
        t[n // 3, :3] = 1e4  # outside the map
        t[n // 2, :3] = room["map"].min  # zero offsets
    return np.ascontiguousarray(t, np.float32)


# workgroups of 4, 8 and 16 poses, their last one ragged, and one past the split form
@pytest.mark.parametrize("n", [1, 3, 4, 5, 2048, 2049, 5632, 5635, 20480, 20481])
def test_poses_at_dispatch_limits(gpu, room, n):
    g, t = _open(gpu, room), _poses(room, n)
    cloud = room["step"].cloud[:300]
    for roll, pitch in ((0.0, 0.0), (0.05, -0.03)):
        w = g.cloud_weights(cloud, t[:, 0], t[:, 1], t[:, 2], t[:, 3], roll, pitch)
        ow = oracle.cloud_weight_batch(room["ogrid"], cloud, t[:, 0], t[:, 1], t[:, 2], t[:, 3], roll, pitch)
        assert np.array_equal(w.view(np.int32), ow.view(np.int32)), (n, roll)


# kernels of every index kind and cell mode; clouds of 0 points, below and
# around one tile (256, 128 and 64 points), two and several tiles
@pytest.mark.parametrize("env", [None, ("A3D_FORCE_IDX64", "1"), ("A3D_FORCE_IDX64", "2"), ("A3D_FORCE_IDX32", "2"),
                                 ("A3D_FORCE_NEAR_TEST", "1")], ids=str)
@pytest.mark.parametrize("n", [37, 2083, 5645])
def test_poses_at_tile_edges(gpu, room, env, n, monkeypatch):
    if env:
        monkeypatch.setenv(*env)
    g, t = _open(gpu, room), _poses(room, n)
    for m in (0, 1, 10, 11, 31, 33, 63, 64, 65, 127, 129, 255, 256, 257, 513, 800):
        cloud = np.ascontiguousarray(room["step"].cloud[:m])
        if m > 20:
            cloud = cloud.copy()
            cloud[m - 3] = np.nan
            cloud[m // 2, 1] = np.inf
        w = g.cloud_weights(cloud, t[:, 0], t[:, 1], t[:, 2], t[:, 3])
        ow = oracle.cloud_weight_batch(room["ogrid"], cloud, t[:, 0], t[:, 1], t[:, 2], t[:, 3])
        assert np.array_equal(w.view(np.int32), ow.view(np.int32)), (n, m)


# whole turns of 16,384 by whole-cloud wavefronts and the rest split: no rest, the
# smallest, the largest split one, one more; clouds around the rule's 2,048 points
@pytest.mark.parametrize("n,m", [(32768, 2050), (32769, 2050), (34816, 2050), (34817, 2050), (32900, 2047), (32900, 2048)])
def test_rest_of_a_turn(gpu, room, n, m):
    g, t = _open(gpu, room), _poses(room, n)
    cloud = np.resize(room["step"].cloud, (m, 3)).astype(np.float32)
    w = g.cloud_weights(cloud, t[:, 0], t[:, 1], t[:, 2], t[:, 3])
    ow = oracle.cloud_weight_batch(room["ogrid"], cloud, t[:, 0], t[:, 1], t[:, 2], t[:, 3])
    assert np.array_equal(w.view(np.int32), ow.view(np.int32))


# whole-cloud wavefronts: the last tile's rest, at every tile and wavefront shape
@pytest.mark.parametrize("ppw", [16, 32, 64])
@pytest.mark.parametrize("tile", [32, 256])
def test_last_tile_of_whole_cloud_wavefronts(gpu, room, ppw, tile):
    g, t = _open(gpu, room), _poses(room, 21000)
    saved = gpu.get_tile(), gpu.get_cloud_tile()
    try:
        gpu.set_tile(ppw)
        gpu.set_cloud_tile(tile)
        for m in (0, 1, 7, 8, 9, 15, 16, 17, 31, 32, 33, 255, 256, 257, 300):
            cloud = np.ascontiguousarray(room["step"].cloud[:m])
            w = g.cloud_weights(cloud, t[:, 0], t[:, 1], t[:, 2], t[:, 3])
            ow = oracle.cloud_weight_batch(room["ogrid"], cloud, t[:, 0], t[:, 1], t[:, 2], t[:, 3])
            assert np.array_equal(w.view(np.int32), ow.view(np.int32)), m
    finally:
        gpu.set_tile(saved[0])
        gpu.set_cloud_tile(saved[1])
