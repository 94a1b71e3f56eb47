"""The allocation-free entry point's grids: its static array is a fixed size, so the
workspace of a large grid must not grow.  A grid of whole-workgroup members needs at
most 164 bytes a workgroup (level-set words, parameter and budget partials, each for
two member slots) besides the member and argument words."""
import pytest

from jcm_amd import _native


@pytest.mark.parametrize("nlon,nlat,nmember", [(1280, 640, 1), (1280, 640, 7), (640, 320, 30), (512, 256, 3), (96, 48, 300)])
def test_large_grids_keep_their_workspace(nlon, nlat, nmember):
    lib = _native.load()
    blocks = -(-nlon * nlat * nmember // 256)
    need = lib.speedy_workspace_bytes(nlon, nlat, nmember)
    assert 0 < need <= 164 * blocks + 8192 + 8 * nmember
    assert need <= lib.speedy_noalloc_max_bytes()
