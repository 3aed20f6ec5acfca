"""shade (image and gradients) at the edges of its pixel passes' 30x14 inner
tiles, for every way of passing the attributes (three channels are a compiled
case, other counts a run-time one), against the FP64 reference in float64.

Bounds: everything is float64 with the reference's own formulas; sums of a few
thousand terms in another order, and the antialiasing edge term's conditioning
(about 1e4 here), leave 1e-10 of the norm."""
import numpy as np
import pytest
import torch

import oracle
from vk_gltf_viewer_amd import diff as D
from vk_gltf_viewer_amd.scene import view_desc

pytestmark = pytest.mark.gpu


def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("fused", [True, False])
@pytest.mark.parametrize("height,width,channels", [(1, 2, 3), (13, 29, 3), (14, 30, 1), (15, 31, 3), (28, 60, 4),
                                                   (29, 61, 8), (64, 5, 2), (3, 100, 3)])
def test_tile_edges(height, width, channels, fused):
    s = D.c4_scene(instances=2, cameras=2, size=32, frequency=6)
    vps = np.stack([D.camera_matrix(view_desc(width, height, (1.1 + 0.2 * k, 0.2, 0.9), (1.1, 0.0, 0.0), fovy_deg=40.0))
                    for k in range(2)])
    clip = D.clip_positions(_t(s.pos).double(), _t(s.xforms).double(), _t(vps).double())
    tris = _t(s.tris)
    e = D.ext()
    ids, depth = e.rasterize(clip.float().contiguous(), tris, height, width, False)
    rng = np.random.default_rng(height * 1000 + width)
    attr, target = rng.random((len(s.pos), channels)), rng.random((2, height, width, channels))
    c, a = clip.clone().requires_grad_(), _t(attr).requires_grad_()
    img = e.shade(c, a, tris, ids, depth) if fused else e.antialias(e.interpolate(c, a, tris, ids), c, tris, ids, depth)
    ((img - _t(target)) ** 2).sum().backward()
    args = (clip.cpu().numpy(), attr, s.tris, ids.cpu().numpy(), depth.cpu().numpy(), target)
    _, ref = oracle.diff_forward(*args)
    g_clip, g_attr = oracle.diff_backward(*args, True)
    assert (ids > 0).any()
    err = np.abs(img.detach().cpu().numpy() - ref).max()
    gc = np.linalg.norm(c.grad.cpu().numpy() - g_clip) / np.linalg.norm(g_clip)
    ga = np.linalg.norm(a.grad.cpu().numpy() - g_attr) / np.linalg.norm(g_attr)
    print(f"{height}x{width}x{channels} fused {fused}: image {err:.1e}, clip {gc:.1e}, attr {ga:.1e}", flush=True)
    assert err <= 1e-10 and gc <= 1e-10 and ga <= 1e-10
