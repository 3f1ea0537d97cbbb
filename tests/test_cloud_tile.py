"""CPU: the cloud tile's setting and the tile single-filter and pose launches
stage, which is their own until a tile other than the default is set."""
import pytest

from amcl3d_amd import _lib, autotune


def _single():
    return _lib.load()._ZN3a3d12single_chunkEv()  # a3d::single_chunk()


@pytest.mark.parametrize("tile", [32, 64, 128, 256])
def test_saving_and_restoring_the_tile_changes_nothing(tile):
    shape, single = autotune.get_shape(), _single()
    saved = _lib.get_cloud_tile()
    _lib.set_cloud_tile(saved)
    assert (_lib.get_cloud_tile(), _single()) == (saved, single)
    _lib.set_cloud_tile(tile)
    assert _lib.get_cloud_tile() == tile
    if tile != 64:
        assert _single() == tile
    _lib.set_cloud_tile(saved)
    assert (_lib.get_cloud_tile(), _single()) == (saved, single)
    autotune.set_shape((0, 16, 1, tile))
    autotune.set_shape(shape)
    assert (autotune.get_shape(), _single()) == (shape, single)
