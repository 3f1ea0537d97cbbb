"""predict's host draws on both sides of the sizes where they are read in place
(4,096 particles) and copied through pinned memory (65,536): bit for bit."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu
F32 = np.float32


@pytest.mark.parametrize("n", [4096, 4097, 65536, 65537, 200000])
def test_draws(gpu, n):
    rng = np.random.default_rng(n)
    p = rng.uniform(0, 1, (n, 7)).astype(F32)
    z4 = rng.standard_normal((n, 4)).astype(F32)
    pf = gpu.ParticleFilter()
    pf.set_particles(p)
    mods, d = (0.1, 0.2, 0.3, 0.4), (0.1, -0.2, 0.05, 0.02)
    pf.predict(*mods, *d, z4)
    assert np.array_equal(pf.particles().view(np.int32), oracle.pf_predict(p, mods, d, z4).view(np.int32))
