"""Pixel slots of small triangles: meshlets whose slot counts and live-triangle
counts lie at the edges of the wave's scans (1, 63, 64, 65 and 124 triangles),
light ones (at most one slot a lane), heavy ones whose slots are deferred and,
with more of them than the staging holds, heavy ones that walk thousands of
slots a lane.  Keys and colours equal the oracle's."""
import numpy as np
import pytest

import oracle
from gltfgen import Builder
from vk_gltf_viewer_amd import _native as N
from vk_gltf_viewer_amd import gltf
from vk_gltf_viewer_amd.renderer import Renderer
from vk_gltf_viewer_amd.scene import camera_from_view, view_desc

pytestmark = pytest.mark.gpu

W, H = 331, 217


def clusters(tmp_path, triangles, copies, extent):
    """`copies` meshes of `triangles` random triangles over 64 vertices in a
    cube of side `extent`, at random places before the camera."""
    rng = np.random.default_rng(1000 * triangles + copies)
    b = Builder()
    roots = []
    m = b.material([0.7, 0.5, 0.3, 1.0], double_sided=True)
    for _ in range(copies):
        pos = ((rng.random((64, 3)) - 0.5) * extent).astype(np.float32)
        idx = np.stack([rng.permutation(64)[:3] for _ in range(triangles)]).astype(np.uint32)
        mesh = b.mesh([{"attributes": {"POSITION": b.accessor(pos, minmax=True)},
                        "indices": b.accessor(idx.reshape(-1, 1)), "material": m}])
        roots.append(b.node(mesh=mesh, translation=[float(v) for v in rng.uniform((-2, -1.2, -1), (2, 1.2, 1))]))
    b.scene(roots)
    p = tmp_path / "clusters.glb"
    b.write_glb(p)
    return gltf.load_gltf(str(p))


@pytest.mark.parametrize("triangles,copies,extent,small", [
    (1, 1, 0.3, 16), (1, 40, 0.02, 16), (63, 9, 0.1, 16), (64, 9, 0.25, 16), (65, 9, 0.25, 64),
    (124, 9, 0.03, 16), (124, 9, 1.2, 64), (124, 300, 1.2, 64), (124, 300, 1.2, 16),
])
def test_slots_match_the_oracle(tmp_path, triangles, copies, extent, small):
    print(f"{copies} clusters of {triangles} triangles, extent {extent}, small below {small} px", flush=True)
    sc = clusters(tmp_path, triangles, copies, extent)
    cam = camera_from_view(view_desc(W, H, (0.0, 0.0, 5.0), (0.0, 0.0, 0.0), fovy_deg=50.0, znear=0.1))
    _, _, total = oracle.pyramid_info(W, H)
    rk, rc, _ = oracle.frame_reference(oracle.Scene(sc), cam, W, H, N.MODE_REFERENCE, np.zeros(total, np.float32))
    assert (oracle.keys_ids(rk) != 0xFFFFFFFF).any()
    r = Renderer()
    try:
        r.load(sc)
        r.set_tuning(small, 3, 8, 8192)
        view = r.create_view(W, H)
        view.render(cam, N.MODE_REFERENCE)
        assert np.array_equal(view.keys(), rk) and np.array_equal(view.color(), rc)
        view.close()
    finally:
        r.close()
