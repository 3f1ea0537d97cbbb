"""The particle counts around one turn of whole-cloud workgroups, where single
filters and poses change from the split form to them and back, for clouds on
both sides of the rest-of-a-turn rule: bit-exact against the oracle."""
import numpy as np
import pytest

import oracle
from test_gpu_split import _open, _poses, room  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [12288, 12289, 16384, 16385, 16640, 16641])
@pytest.mark.parametrize("m", [200, 2050])
def test_poses_around_a_turn(gpu, room, n, m):  # noqa: F811
    g, t = _open(gpu, room), _poses(room, n)
    cloud = np.resize(room["step"].cloud, (m, 3)).astype(np.float32)
    w = g.cloud_weights(cloud, t[:, 0], t[:, 1], t[:, 2], t[:, 3])
    ow = oracle.cloud_weight_batch(room["ogrid"], cloud, t[:, 0], t[:, 1], t[:, 2], t[:, 3])
    assert np.array_equal(w.view(np.int32), ow.view(np.int32))
