"""The synchronous calls where no pinned host memory can be had: they fall back
on device memory and plain copies, with the same bits.  One child process runs
them with A3D_NO_PINNED=1, which the library reads once."""
import os
import subprocess
import sys

import numpy as np
import pytest

import oracle
from amcl3d_amd import _lib, workloads as W

pytestmark = pytest.mark.gpu
F32 = np.float32
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _calls(gpu):
    out = []
    c = W.room_case(2)
    bm, s, t = c["map"], c["step"], c["particles"][:900]
    grid = gpu.Grid3d()
    grid.open(bm.points(), bm.min, bm.max, bm.res, c["sensor_dev"])
    out.append(grid.read_cells())
    out.append(grid.cloud_weights(s.cloud, t[:, 0], t[:, 1], t[:, 2], t[:, 3]))
    rng = np.random.default_rng(3)
    scan = rng.uniform(-3, 3, (4000, 3)).astype(F32)
    scan[:1500] = scan[:1500] % F32(0.2)  # a crowded voxel
    out.append(_lib.voxel_grid(scan, 0.3))
    pf = gpu.ParticleFilter()
    out.append(pf.getMean())
    for n in (64, 900):
        pf.set_particles(t[:n])
        out.append(pf.getMean())
        pf.predict(0.1, 0.1, 0.1, 0.1, 0.05, 0.01, 0.0, 0.02, rng.standard_normal((n, 4)).astype(F32))
        pf.update(grid, s.cloud, s.ranges, s.alpha, s.sigma)
        out += [pf.getMean(), pf.particles(), pf.resample(0.3, gpu.RESAMPLE_REFERENCE, return_indices=True)]
        pf.update(None, s.cloud, s.ranges, s.alpha, s.sigma)
        out += [pf.getMean(), pf.particles()]
    return out


def test_calls_without_pinned_memory(gpu, tmp_path):
    path = str(tmp_path / "out.npz")
    code = ("import sys; sys.path[:0] = [%r, %r]; import numpy as np, amcl3d_amd as g; g.load();"
            "import test_gpu_no_pinned as t; np.savez(%r, *t._calls(g))" % (ROOT, os.path.join(ROOT, "tests"), path))
    r = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, A3D_NO_PINNED="1"), capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    ref = _calls(gpu)
    with np.load(path) as z:
        assert len(z.files) == len(ref)
        for k, want in enumerate(ref):
            got = z["arr_%d" % k]
            assert got.dtype == want.dtype and got.shape == want.shape, k
            assert got.tobytes() == want.tobytes(), k
    assert np.array_equal(ref[2].view(np.int32), _ref_scan().view(np.int32))


def _ref_scan():
    rng = np.random.default_rng(3)
    scan = rng.uniform(-3, 3, (4000, 3)).astype(F32)
    scan[:1500] = scan[:1500] % F32(0.2)
    return oracle.voxel_grid(scan, 0.3, order_mode=1)
