"""The exact sums, the update tail and resample of filters that one workgroup
takes, at the sizes where their sub-tiles (64), chunks (8,192), fused kernels
(1,024 and 2,048) and dispatch limits end: bit for bit against the oracle."""
import numpy as np
import pytest

import oracle
from amcl3d_amd import workloads as W
from amcl3d_amd.fleet import Fleet

pytestmark = pytest.mark.gpu
F32 = np.float32


@pytest.fixture(scope="module")
def room(gpu):
    c = W.room_case(6)
    bm = c["map"]
    _, prob = oracle.compute_grid(bm.points(), bm.min, bm.max, bm.res, c["sensor_dev"], exp_mode=1)
    return dict(case=c, bm=bm, prob=prob)


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1023, 1024, 1025, 2047, 2048, 2049, 4097, 8192, 8193, 16385, 24575, 24576])
def test_full_step(gpu, room, n):
    """Yaws on both sides of 0 and a map at negative x (mean terms of either sign)."""
    c, bm, s = room["case"], room["bm"], room["case"]["step"]
    rng = np.random.default_rng(n)
    sh = np.array([-10.0, 0.0, 0.0])
    grid = gpu.Grid3d().from_cells(room["prob"], bm.min + sh, bm.max + sh, bm.res, c["sensor_dev"])
    og = oracle.GridMeta(bm.min + sh, bm.max + sh, bm.res, room["prob"])
    parts = W.particles_around(np.array([0.0, 10.0, 1.5, 0.0]), n, rng)
    parts[: n // 50, 2] = -50.0  # some outside the map
    z4 = rng.standard_normal((n, 4)).astype(F32)
    cloud = s.cloud[:200]
    pf = gpu.ParticleFilter()
    pf.set_particles(parts)
    pf.predict(*s.mods, *s.deltas, z4)
    pf.update(grid, cloud, s.ranges, s.alpha, s.sigma)
    upd, mean = pf.particles(), pf.getMean()
    idx = pf.resample(s.u01, gpu.RESAMPLE_REFERENCE, return_indices=True)
    op = oracle.pf_predict(parts, s.mods, s.deltas, z4)
    op, om = oracle.pf_update(op, og, cloud, s.ranges, s.alpha, s.sigma)
    oq, oidx = oracle.pf_resample(op, s.u01, 0)
    assert np.array_equal(upd.view(np.int32), op.view(np.int32))
    assert np.array_equal(mean.view(np.int32), om.view(np.int32))
    assert np.array_equal(idx, oidx)
    assert np.array_equal(pf.particles().view(np.int32), oq.view(np.int32))


KINDS = {
    "exponential": lambda n, r: r.exponential(1.0, n),
    "growing": lambda n, r: np.exp(np.linspace(-40, 10, n)),
    "ties": lambda n, r: r.integers(0, 8, n) * 2.0 ** -20,
    "equal": lambda n, r: np.full(n, 1.0 / n),
    "zeros first": lambda n, r: np.concatenate([np.zeros(n // 2), r.uniform(0, 1, n - n // 2)]),
    "subnormal": lambda n, r: r.uniform(0, 1, n) * 1e-41,
    "one hot": lambda n, r: np.eye(1, n, 2 * n // 3)[0],
    "nan": lambda n, r: np.where(np.arange(n) == n // 2, np.nan, r.uniform(0, 1, n)),
    "inf": lambda n, r: np.where(np.arange(n) == n // 2, np.inf, r.uniform(0, 1, n)),
    "negative run": lambda n, r: r.uniform(0, 1, n) * np.where(np.abs(np.arange(n) - n // 2) < n // 9, -1, 1),
}


@pytest.mark.parametrize("n", [700, 2048, 2049, 8192, 20000])
@pytest.mark.parametrize("kind", list(KINDS))
def test_resample_running_sum(gpu, kind, n):
    p = np.zeros((n, 7), F32)
    p[:, 0] = np.arange(n)
    p[:, 4] = KINDS[kind](n, np.random.default_rng(3)).astype(F32)
    pf = gpu.ParticleFilter()
    pf.set_particles(p)
    idx = pf.resample(0.41, gpu.RESAMPLE_REFERENCE, return_indices=True)
    assert np.array_equal(idx, oracle.resample_indices(p[:, 4], 0.41, 0)), kind
    assert np.array_equal(pf.particles()[:, 0], p[idx, 0])


@pytest.mark.parametrize("n", [1, 1023, 1024, 1025, 5000, 70000, 1_100_000])
def test_fp64_prefix(gpu, n):
    """One workgroup per block of 1,024, the earlier blocks' totals in order (more than 1,024 of them at the last size)."""
    p = np.zeros((n, 7), F32)
    p[:, 4] = np.random.default_rng(n).exponential(1.0, n).astype(F32)
    p[:, 4] /= p[:, 4].sum(dtype=np.float64)
    pf = gpu.ParticleFilter()
    pf.set_particles(p)
    idx = pf.resample(0.23, gpu.RESAMPLE_FP64, return_indices=True)
    assert np.array_equal(idx, oracle.resample_indices(p[:, 4], 0.23, 1))


@pytest.mark.parametrize("largest", [1000, 2000, 2100])
def test_fleet_of_small_filters(gpu, room, largest):
    c, bm, s = room["case"], room["bm"], room["case"]["step"]
    grid = gpu.Grid3d().from_cells(room["prob"], bm.min, bm.max, bm.res, c["sensor_dev"])
    og = oracle.GridMeta(bm.min, bm.max, bm.res, room["prob"])
    counts = [1, 64, 333, largest]
    rng = np.random.default_rng(largest)
    parts = [W.particles_around(np.array([10.0, 10.0, 1.5, 0.1 * n]), n, rng) for n in counts]
    fl = Fleet(counts)
    fl.set_particles(np.concatenate(parts))
    F = len(counts)
    fl.stage_update([s.cloud[:120]] * F, [s.ranges] * F, s.alpha, s.sigma)
    fl.update_staged(grid)
    means = fl.means()
    u = np.linspace(0.1, 0.9, F).astype(F32)
    fl.resample(u)
    got, at = fl.particles(), 0
    for k, n in enumerate(counts):
        op, om = oracle.pf_update(parts[k], og, s.cloud[:120], s.ranges, s.alpha, s.sigma)
        oq, _ = oracle.pf_resample(op, float(u[k]), 0)
        assert np.array_equal(means[k].view(np.int32), om.view(np.int32)), n
        assert np.array_equal(got[at:at + n].view(np.int32), oq.view(np.int32)), n
        at += n
