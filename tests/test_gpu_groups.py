"""The meshlet raster's batches over several meshlets of a wave: with one block
a CU and more meshlets than waves, a wave takes two, three (a full group), four
or seven and eight of them, with 1, 63, 64, 65 or 124 triangles or none that
holds a pixel centre, in any order (the visible list's order is free).  In one
case each only some meshlets' triangles find the big queue or the clip queue
full, so that single meshlets of a group are redone.  Keys and colours equal
the oracle's."""
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
WAVES = 256 * 4      # one block of four waves on each CU

# triangles and side of the cube they lie in: live ones, none live, ones beyond the small limit
SMALL = [(1, 0.2), (63, 0.2), (64, 0.2), (65, 0.2), (124, 0.2), (124, 1e-4), (1, 1e-4)]
LARGE = [(2, 3.0)]


def crowd(tmp_path, kinds, copies, near):
    rng = np.random.default_rng(copies + len(kinds))
    b = Builder()
    m = b.material([0.7, 0.5, 0.3, 1.0], double_sided=True)
    meshes = []
    for triangles, extent in kinds:
        pos = ((rng.random((64, 3)) - 0.5) * extent).astype(np.float32)
        idx = np.stack([rng.permutation(64)[:3] for _ in range(triangles)]).astype(np.uint32)
        meshes.append(b.mesh([{"attributes": {"POSITION": b.accessor(pos, minmax=True)},
                               "indices": b.accessor(idx.reshape(-1, 1)), "material": m}]))
    # large ones are few; some of them reach behind the camera where `near`
    which = np.where(rng.random(copies) < 0.03, len(kinds) - 1, rng.integers(0, len(kinds) - len(LARGE), copies))
    at = rng.uniform((-2, -1.2, -1), (2, 1.2, 1), (copies, 3))
    at[which == len(kinds) - 1, 2] += 4.6 * near
    b.scene([b.node(mesh=meshes[k], translation=[float(x) for x in v]) for k, v in zip(which, at)])
    p = tmp_path / "crowd.glb"
    b.write_glb(p)
    return gltf.load_gltf(str(p))


@pytest.mark.parametrize("copies,near,caps,overflow", [
    (2 * WAVES, 0.0, {}, 0), (3 * WAVES, 0.0, {}, 0), (3 * WAVES + 500, 0.0, {}, 0), (7 * WAVES + 13, 0.0, {}, 0),
    (3 * WAVES + 500, 0.0, {"big_triangle_capacity": 4}, 1), (3 * WAVES + 500, 1.0, {"clip_triangle_capacity": 4}, 2),
])
def test_groups_match_the_oracle(tmp_path, copies, near, caps, overflow):
    print(f"{copies} meshlets, {caps}", flush=True)
    sc = crowd(tmp_path, SMALL + LARGE, copies, near)
    cam = camera_from_view(view_desc(W, H, (0.0, 0.0, 5.0), (0.0, 0.0, 0.0), fovy_deg=50.0, znear=0.1))
    _, _, total = oracle.pyramid_info(W, H)
    rk, rc, rv = oracle.frame_reference(oracle.Scene(sc), cam, W, H, N.MODE_REFERENCE, np.zeros(total, np.float32))
    assert len(rv) > 0.9 * copies
    r = Renderer(**caps)
    try:
        r.load(sc)
        r.set_tuning(16, 1, 8, 8192)
        view = r.create_view(W, H)
        view.render(cam, N.MODE_REFERENCE)
        st = view.stats()
        print(f"  visible {len(rv)}, big {st.big_triangles}, clipped {st.clipped_triangles}, overflow {st.overflow}", flush=True)
        assert np.array_equal(view.keys(), rk) and np.array_equal(view.color(), rc)
        assert st.overflow & 3 == overflow
        view.close()
    finally:
        r.close()
