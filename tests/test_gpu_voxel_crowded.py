"""VoxelGrid with voxels of more than 1,024 points, which a workgroup each sums:
at the edges of its tiles (1,024 points) and windows (2^18 cloud indices), with
a voxel's points together or scattered in the cloud, bit for bit against the
oracle summing in point order."""
import numpy as np
import pytest

import oracle
from amcl3d_amd import _lib

pytestmark = pytest.mark.gpu
F32 = np.float32


def _cloud(sizes, rng, scattered):
    """sizes[k] points in voxel (2k, 0, 0) of a unit lattice."""
    at = np.repeat(np.arange(len(sizes)) * 2, sizes)
    c = rng.uniform(0.01, 0.99, (len(at), 3)).astype(F32)
    c[:, 0] += at.astype(F32)
    return c[rng.permutation(len(c))] if scattered else c


def _check(c):
    got = _lib.voxel_grid(c, 1.0)
    ref = oracle.voxel_grid(c, 1.0, order_mode=1)
    assert got.shape == ref.shape
    assert np.array_equal(got.view(np.int32), ref.view(np.int32))


@pytest.mark.parametrize("scattered", [False, True])
@pytest.mark.parametrize("sizes", [(1024, 1025, 1), (2047, 2048, 2049, 5), (3000, 1023, 7000, 33), (40000,),
                                   tuple([1100] * 300)], ids=lambda s: "%dx%d" % (len(s), s[0]))
def test_tiles(gpu, sizes, scattered):
    _check(_cloud(sizes, np.random.default_rng(len(sizes)), scattered))


# clouds that end at a window's edge and past it; the points of a voxel in one window, in all, across an edge
@pytest.mark.parametrize("n", [(1 << 18) - 1, 1 << 18, (1 << 18) + 1, (1 << 18) + 40, 700001, 1 << 20])
def test_windows(gpu, n):
    rng = np.random.default_rng(n)
    c = _cloud((n,), rng, False)
    c[:, 0] += 2 * rng.integers(0, 60000, n).astype(F32)  # nearly all on their own
    c[rng.choice(n, 5000, replace=False), 0] = 0.5
    c[n - 1500:, 0] = 4.5
    c[(1 << 18) - 1300:(1 << 18) + 1300, 0] = 8.5
    _check(c)


# workgroups of 1,024 points join their voxels' bits: every point another word, all one word, one ragged workgroup
@pytest.mark.parametrize("n", [1023, 1024, 1025, 5000])
@pytest.mark.parametrize("spread", [1, 33, 64 * 1024])
def test_marks(gpu, n, spread):
    rng = np.random.default_rng(n + spread)
    c = rng.uniform(0.01, 0.99, (n, 3)).astype(F32)
    c[:, 0] += rng.integers(0, spread, n).astype(F32)
    c[::53] = np.nan
    _check(c)
