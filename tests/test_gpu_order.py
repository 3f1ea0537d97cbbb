"""The particle visiting order at the sizes where its kernels change: it
changes no bit of an update, whatever its keys are made of."""
import numpy as np
import pytest

from amcl3d_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def room():
    c = W.room_case(1)
    bm = c["map"]
    pts = bm.points()
    c.update(points=pts)
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


# sorted by one workgroup (1, 4 or 8 particles per thread) and by four kernels;
# sets whose key bits all go to one coordinate, none at all, and a spread one
@pytest.mark.parametrize("n", [2049, 4096, 4097, 8192, 8193, 16385])
def test_visiting_order_changes_no_bit(gpu, room, n):
    g, s = _open(gpu, room), room["step"]
    p = np.zeros((n, 7), np.float32)
    t = _poses(room, n)
    for kind in ("mixed", "equal", "z only", "yaw only", "spread"):
        p[:, :4] = t[0]
        if kind == "mixed":
            p[:, :4] = t
        elif kind == "z only":
            p[:, 2] = t[:, 2]
        elif kind == "yaw only":
            p[:, 3] = np.linspace(-3.1, 3.1, n)
        elif kind == "spread":
            p[:, :2] = np.random.default_rng(n).uniform(0.1, 19.9, (n, 2))
        out = []
        saved = gpu.get_order()
        try:
            for order in (gpu.ORDER_INDEX, gpu.ORDER_SPATIAL):
                gpu.set_order(order)
                pf = gpu.ParticleFilter()
                pf.set_particles(p)
                pf.update(g, s.cloud[:200], s.ranges, s.alpha, s.sigma, 0.0, 0.0)
                out.append(pf.particles())
        finally:
            gpu.set_order(saved)
        assert np.array_equal(out[0].view(np.int32), out[1].view(np.int32)), (n, kind)


# batches: one filter per grid row, uneven ones
@pytest.mark.parametrize("largest", [257, 4000, 20481])
def test_fleet_order_changes_no_bit(gpu, room, largest):
    from amcl3d_amd.fleet import Fleet

    g, s = _open(gpu, room), room["step"]
    counts = [1, 65, largest]
    p = np.zeros((sum(counts), 7), np.float32)
    p[:, :4] = _poses(room, sum(counts))
    fl = Fleet(counts)
    fl.set_particles(p)
    clouds = [s.cloud[:150], s.cloud[:77], s.cloud[:200]]
    fl.stage_update(clouds, [s.ranges] * 3, s.alpha, s.sigma)
    fl.update_staged(g)
    got, at = fl.particles(), 0
    for n, c in zip(counts, clouds):
        pf = gpu.ParticleFilter()
        pf.set_particles(p[at:at + n])
        pf.update(g, c, s.ranges, s.alpha, s.sigma, 0.0, 0.0)
        assert np.array_equal(got[at:at + n].view(np.int32), pf.particles().view(np.int32)), n
        at += n
