"""Readbacks through the pinned stage: sizes around its threshold, its pieces
and its halves, with a partial last piece, equal to the same data read in small
copies; several reads in a row into fresh and reused memory."""
import numpy as np
import pytest

from vk_gltf_viewer_amd import _native as N
from vk_gltf_viewer_amd.renderer import Renderer

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rend():
    r = Renderer()
    yield r
    r.close()


# 64-byte matrices: 64 KB is 1024 of them, a piece 256, a half 32768
@pytest.mark.parametrize("count", [1, 1023, 1024, 1025, 4096 + 255, 32768, 32769, 3 * 32768 + 257])
def test_transforms(rend, count):
    want = np.random.default_rng(count).normal(size=(count, 16)).astype(np.float32)
    rend.set_transforms(want)
    for _ in range(3):
        assert np.array_equal(rend.read_transforms(count), want)
    part = max(1, count - 3)          # a prefix, ending inside a piece
    assert np.array_equal(rend.read_transforms(part), want[:part])


@pytest.mark.parametrize("width,height", [(2, 1), (181, 91), (640, 360), (1027, 771)])
def test_pyramid_and_keys(rend, width, height):
    v = rend.create_view(width, height)
    try:
        texels = np.random.default_rng(width).random(v.pyramid_texels).astype(np.float32)
        v.write_pyramid(texels)
        assert np.array_equal(v.pyramid(), texels)
        depth = np.random.default_rng(height).random((height, width)).astype(np.float32)
        v.write_depth(depth)
        ids, got = v.ids_depth()
        assert np.array_equal(got, depth) and np.all(ids == N.VISBUFFER_CLEAR)
    finally:
        v.close()
