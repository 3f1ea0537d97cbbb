"""VoxelGrid's bitmap ranking and its sort, at the sizes where their lists,
workgroups and dispatch limits end, bit for bit against the oracle summing in
point order."""
import numpy as np
import pytest

import oracle
from amcl3d_amd import _lib

pytestmark = pytest.mark.gpu
F32 = np.float32


def _check(c, leaf):
    got = _lib.voxel_grid(c, leaf)
    ref = oracle.voxel_grid(c, leaf, order_mode=1)
    assert got.shape == ref.shape
    assert np.array_equal(got.view(np.int32), ref.view(np.int32))


@pytest.mark.parametrize("n", [1, 2, 31, 33, 63, 65, 255, 257, 1023, 1025, 30001])
def test_sizes(gpu, n):
    rng = np.random.default_rng(n)
    _check(rng.uniform(-3, 3, (n, 3)).astype(F32), 0.25)


# points per voxel: below, at and above 32 (half a wavefront), ranked by a
# wavefront, past 1,024 and past sqrt(2 n) (searched), all in one voxel
@pytest.mark.parametrize("per,voxels", [(31, 50), (32, 50), (33, 50), (64, 40), (65, 40), (300, 200), (700, 3), (1024, 700),
                                        (1025, 9), (20000, 1)])
def test_crowded_voxels(gpu, per, voxels):
    rng = np.random.default_rng(per)
    at = np.repeat(rng.permutation(voxels * 3)[:voxels], per)
    c = rng.uniform(0.01, 0.99, (voxels * per, 3)).astype(F32) * F32(0.5)
    c[:, 0] += at.astype(F32) * F32(0.5)
    c = c[rng.permutation(len(c))]
    c[:: max(2, len(c) // 5)] += F32(7.0)  # some on their own
    _check(c, 0.5)


# lattices around the bitmap's limit (2^26 voxels), a flat one, one far from the
# origin, and points without a voxel
@pytest.mark.parametrize("ext", [(403.0, 403.0, 412.0), (406.0, 406.0, 408.0), (1300.0, 1300.0, 1200.0), (60000.0, 0.0, 3.0)])
def test_lattices(gpu, ext):
    rng = np.random.default_rng(7)
    c = (rng.uniform(0, 1, (5000, 3)) * np.array(ext)).astype(F32)
    c[0], c[1] = 0.0, np.array(ext, F32)
    c[5::50] = np.nan
    c[9, 1] = np.inf
    _check(c, 1.0)
    _check(c + np.array([1e5, -3e5, 10.0], F32), 1.0)


def test_more_points_than_the_bitmap_takes(gpu):
    rng = np.random.default_rng(3)
    c = rng.uniform(-20, 20, ((1 << 20) + 1, 3)).astype(F32)
    _check(c, 0.5)
    _check(c[:-1], 0.5)
