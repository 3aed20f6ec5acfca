"""vkgv_view_aa_image_noalloc against the FP64 reference fed the same keys, into
an image filled with NaN, views of part of a tile to many (bound as in
test_gpu_aa_tiles.py: one double rounded to float32)."""
import numpy as np
import pytest
import torch

import oracle
from vk_gltf_viewer_amd import _native as N
from vk_gltf_viewer_amd.renderer import Renderer
from vk_gltf_viewer_amd.scene import Scene, camera_from_view, view_desc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height", [(5, 3), (65, 9), (320, 180), (641, 363)])
def test_image_matches_the_reference(width, height):
    sc = Scene(1, 1, 64).arrays()
    r = Renderer()
    try:
        r.load(sc)
        cam = camera_from_view(view_desc(width, height, (0.0, 15.0, 90.0), (0.0, 0.0, 0.0), fovy_deg=45.0))
        view = r.create_view(width, height)
        view.render(cam, N.CULL_FRUSTUM | N.CULL_TWO_PASS)
        out = torch.full((height, width, 3), float("nan"), device="cuda")
        view.aa_image_noalloc(cam, out)
        ref = oracle.frame_aa_image(oracle.Scene(sc), np.asarray(cam.view_projection, np.float32), view.keys(), width, height)
        err = np.abs(out.cpu().numpy() - ref).max()
        print(f"{width}x{height}: {err:.1e}", flush=True)
        assert err <= 1e-7 and (ref.any() or width < 64)   # the smallest view may show no sphere
        view.close()
    finally:
        r.close()
