"""The calls' pooled buffers: threads that take and give them back side by side,
sizes on both sides of the pinned paths' limits, and state that outlives a call."""
import threading

import numpy as np
import pytest

import oracle
from amcl3d_amd import _lib, workloads as W

pytestmark = pytest.mark.gpu
F32 = np.float32


def test_threads_share_the_pool(gpu):
    c = W.room_case(2)
    bm, s = c["map"], c["step"]
    pts = bm.points()
    _, prob = oracle.compute_grid(pts, bm.min, bm.max, bm.res, c["sensor_dev"], exp_mode=1)
    og = oracle.GridMeta(bm.min, bm.max, bm.res, prob)
    failed = []

    def work(k):
        try:
            rng = np.random.default_rng(k)
            grid = gpu.Grid3d().from_cells(prob, bm.min, bm.max, bm.res, c["sensor_dev"])
            for r in range(12):
                n, m = int(rng.integers(1, 5000)), int(rng.integers(1, 400))
                t = c["particles"][rng.integers(0, len(c["particles"]), n)]
                w = grid.cloud_weights(s.cloud[:m], t[:, 0], t[:, 1], t[:, 2], t[:, 3])
                ow = oracle.cloud_weight_batch(og, s.cloud[:m], t[:, 0], t[:, 1], t[:, 2], t[:, 3], nthreads=1)
                assert np.array_equal(w.view(np.int32), ow.view(np.int32))
                v = rng.uniform(-2, 2, (int(rng.integers(1, 3000)), 3)).astype(F32)
                assert np.array_equal(_lib.voxel_grid(v, 0.3), oracle.voxel_grid(v, 0.3, order_mode=1))
                p = rng.uniform(0, 1, (n, 7)).astype(F32)
                pf = gpu.ParticleFilter()
                pf.set_particles(p)
                assert np.array_equal(pf.particles(), p)
        except Exception as e:  # noqa: BLE001
            failed.append((k, repr(e)))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed


# draws read in place and copied (4,096); rows, draws and indices past the
# pinned paths' 16 MiB (599,186 rows of seven floats; 1,048,576 draws of four)
@pytest.mark.parametrize("n", [1, 4096, 4097, 599186, 599187, 1048577])
def test_rows_draws_and_indices(gpu, n):
    rng = np.random.default_rng(n)
    p = rng.uniform(0, 1, (n, 7)).astype(F32)
    p[:, 4] = 1.0 / n
    z4 = rng.standard_normal((n, 4)).astype(F32)
    pf = gpu.ParticleFilter()
    pf.set_particles(p)
    assert np.array_equal(pf.particles(), p)
    mods, d = (0.1, 0.2, 0.3, 0.4), (0.1, -0.2, 0.05, 0.02)
    pf.predict(*mods, *d, z4)
    op = oracle.pf_predict(p, mods, d, z4)
    assert np.array_equal(pf.particles().view(np.int32), op.view(np.int32))
    idx = pf.resample(0.3, gpu.RESAMPLE_REFERENCE, return_indices=True)
    assert np.array_equal(idx, oracle.resample_indices(op[:, 4], 0.3, 0))


def test_mean_follows_resizes_and_updates(gpu):
    c = W.room_case(2)
    bm, s = c["map"], c["step"]
    grid = gpu.Grid3d()
    grid.open(bm.points(), bm.min, bm.max, bm.res, c["sensor_dev"])
    pf = gpu.ParticleFilter()
    assert not pf.getMean().any()
    for n in (64, 900, 64):
        pf.set_particles(c["particles"][:n])
        assert not pf.getMean().any()  # a resized set has no mean yet
        pf.update(grid, s.cloud, s.ranges, s.alpha, s.sigma)
        m = pf.getMean()
        q = pf.particles()
        assert np.allclose(m, (q[:, 4:5].astype(np.float64) * q[:, :4]).sum(0), rtol=1e-4, atol=1e-5)
        pf.update(None, s.cloud, s.ranges, s.alpha, s.sigma)
        assert not pf.getMean().any()
