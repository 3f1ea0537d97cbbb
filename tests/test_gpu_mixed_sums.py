"""The mean's sums over terms of both signs: runs of mixed sub-tiles of 64 that
begin, end and go on where the walk's windows of 64 sub-tiles do, between
sub-tiles of one sign and of zeros, at one to three chunks of 8,192: bit for bit
against the oracle."""
import numpy as np
import pytest

import oracle
from amcl3d_amd import workloads as W

pytestmark = pytest.mark.gpu
F32 = np.float32


def _signs(kind, n, rng):
    q = np.arange(n) // 64
    s = rng.choice([-1.0, 1.0], n)
    if kind == "all mixed":
        return s
    if kind == "one sign, then mixed":
        return np.where(q < 64, 1.0, s)
    if kind == "zeros, then mixed":
        return np.where(q < 64, 0.0, s)
    if kind == "alternating":
        return np.where(q % 2 == 0, np.where(q % 4 == 0, 1.0, -1.0), s)
    return np.where(np.isin(q % 67, (0, 1, 62, 63, 64)), -1.0, s)  # single-signed ones around the windows' edges


@pytest.mark.parametrize("kind", ["all mixed", "one sign, then mixed", "zeros, then mixed", "alternating", "edges"])
@pytest.mark.parametrize("n", [2049, 4097, 8193, 20000])
def test_mean_of_both_signs(gpu, kind, n):
    c = W.room_case(6)
    bm, s = c["map"], c["step"]
    _, prob = oracle.compute_grid(bm.points(), bm.min, bm.max, bm.res, c["sensor_dev"], exp_mode=1)
    sh = np.array([-10.0, -10.0, 0.0])
    grid = gpu.Grid3d().from_cells(prob, bm.min + sh, bm.max + sh, bm.res, c["sensor_dev"])
    og = oracle.GridMeta(bm.min + sh, bm.max + sh, bm.res, prob)
    rng = np.random.default_rng(n)
    p = np.zeros((n, 7), F32)
    p[:, 0] = rng.uniform(0.01, 9, n) * _signs(kind, n, rng)
    p[:, 1] = rng.uniform(0.01, 9, n) * _signs(kind, n, rng)
    p[:, 2] = rng.uniform(0.5, 4, n)
    p[:, 3] = rng.uniform(0.01, 3.1, n) * _signs(kind, n, rng)
    pf = gpu.ParticleFilter()
    pf.set_particles(p)
    pf.update(grid, s.cloud[:60], s.ranges, s.alpha, s.sigma)
    op, om = oracle.pf_update(p, og, s.cloud[:60], s.ranges, s.alpha, s.sigma)
    assert np.array_equal(pf.particles().view(np.int32), op.view(np.int32))
    assert np.array_equal(pf.getMean().view(np.int32), om.view(np.int32))
