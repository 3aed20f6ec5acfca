"""Texel wrap at the ends of its range: texture sides of 1, odd and 16384
texels, coordinates of a texel or less, up to 2^30 texels and beyond (where they
are cut), on both sides of zero, under every wrap mode, colours equal to the
oracle's."""
import numpy as np
import pytest

import oracle
from test_gpu_parity import compare_keys
from texscene import quad_scene
from vk_gltf_viewer_amd import _native as N
from vk_gltf_viewer_amd.renderer import Renderer
from vk_gltf_viewer_amd.scene import Texture

pytestmark = pytest.mark.gpu

W, H = 97, 61


@pytest.fixture(scope="module")
def rend():
    r = Renderer()
    yield r
    r.close()


@pytest.mark.parametrize("wrap", [N.WRAP_REPEAT, N.WRAP_MIRRORED_REPEAT, N.WRAP_CLAMP_TO_EDGE])
@pytest.mark.parametrize("sides,scale,offset", [
    ((1, 1), (3.0, -2.0), (0.25, -0.75)), ((16384, 1), (1.0, 5.0), (-0.5, 0.5)), ((1, 16384), (0.01, -2.0), (7.0, 1.0)),
    ((3, 5), (1.0e6, -1.0e6), (-5.0e5, 5.0e5)), ((16384, 7), (65536.0, 3.0e8), (-32768.0, -1.5e8)),
    ((7, 16383), (-4.0e8, 1.0e5), (2.0e8, -65536.0)), ((255, 256), (1.0e20, -1.0e30), (0.0, 1.0)),
])
def test_wrap_matches_oracle(rend, sides, scale, offset, wrap):
    rng = np.random.default_rng(sides[0] + sides[1])
    tex = rng.integers(0, 256, (sides[1], sides[0], 4)).astype(np.uint8)
    sc, cam = quad_scene(W, H, Texture(tex, wrap, wrap), uv_offset=offset, uv_scale=scale)
    print(f"{sides[0]}x{sides[1]} texels, scale {scale}, offset {offset}, wrap {wrap}", flush=True)
    rend.load(sc)
    v = rend.create_view(W, H)
    try:
        flags = N.CULL_FRUSTUM | N.RESOLVE_TEXTURED
        _, _, total = oracle.pyramid_info(W, H)
        rk, rc, _ = oracle.frame_reference(oracle.Scene(sc), cam, W, H, flags, np.zeros(total, np.float32))
        v.render(cam, flags)
        compare_keys(v.keys(), rk, "quad")
        assert len(np.unique(rc)) > 1 or sides == (1, 1) or max(scale) > 1e9
        assert np.array_equal(v.color(), rc)
    finally:
        v.close()
