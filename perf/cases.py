"""The timed workloads: what programs built on this package have it do, through
its public entry points (Renderer, View, Batch, DifferentiableFrame, diff.render).

Kinds
  view     one view's frame (cull, raster, Hi-Z, resolve), and its antialiased
           linear image on the device
  still    one small frame read back to the host, as a thumbnail service does
  cut      a camera cut: history reset, then a few frames of a moving camera
  player   an animated, textured scene: transform update, textured frame with
           motion vectors, colour and motion read back
  views    many views of uneven size as one captured batch frame, and each
           view's image
  pose     images of several views and their gradient to the instance transforms
  fit      the differentiable renderer: image, ids and the gradients to
           positions, albedo and transforms, in each precision
  preview  the same without gradients (evaluation)
  animate  the device transform update, matrices read back

Everything a case needs is made from its seed.  `exact` gives the values of
fit, preview and animate in 64 bits, written in torch and numpy alone; the
frames' images depend on the whole renderer and have none.
"""
from __future__ import annotations

import dataclasses
import functools
import math

import numpy as np
import torch

from vk_gltf_viewer_amd import _native as N
from vk_gltf_viewer_amd import diff as D
from vk_gltf_viewer_amd.frame_grad import DifferentiableFrame
from vk_gltf_viewer_amd.renderer import Renderer
from vk_gltf_viewer_amd.scene import (ANIM_CHANNEL_DTYPE, ANIM_SAMPLER_DTYPE, NODE_DTYPE, Hierarchy, Scene, Texture,
                                      camera_advance, camera_from_view, view_desc)

TWO_PASS = N.CULL_FRUSTUM | N.CULL_TWO_PASS
MODES = {"reference": N.MODE_REFERENCE, "flat": TWO_PASS, "bary": TWO_PASS | N.RESOLVE_BARY,
         "cone": TWO_PASS | N.CULL_CONE | N.RESOLVE_BARY}


def listed():
    return [
        # a thumbnail of a small scene, on the host when the call returns: latency and launches
        {"name": "still_360p", "kind": "still", "scene": "spheres", "objects": 64, "width": 640, "height": 360,
         "mode": "reference"},
        # an interactive frame of the plain configuration at its own size and mode
        {"name": "view_720p", "kind": "view", "scene": "spheres", "objects": 256, "width": 1280, "height": 720,
         "mode": "reference"},
        # the headline frame: the occlusion-heavy city at 4K, steady camera
        {"name": "view_city_4k", "kind": "view", "scene": "city", "objects": 0, "width": 3840, "height": 2160,
         "mode": "bary"},
        # a cut to a moving camera in the city: a cold frame, then frames with a live late pass; odd size
        {"name": "cut_city_1081", "kind": "cut", "scene": "city", "objects": 0, "width": 1921, "height": 1081,
         "mode": "bary", "frames": 4},
        # a player of an animated, textured scene that hands frames to an encoder on the host
        {"name": "player_720p", "kind": "player", "scene": "spheres", "objects": 256, "width": 1280, "height": 720},
        # shadow cascades, cube faces and cameras of uneven size in one captured launch
        {"name": "views_16", "kind": "views", "scene": "spheres", "objects": 256, "views": 16, "mode": "bary"},
        # pose estimation: transforms of many objects from several small views
        {"name": "pose_8", "kind": "pose", "scene": "spheres", "objects": 256, "views": 8, "width": 640, "height": 480},
        # the uneven stress scene: millions of draws, sub-pixel triangles, views up to 4K, with its backward
        {"name": "pose_uneven_4", "kind": "pose", "scene": "uneven", "objects": 3, "views": 4, "width": 3840,
         "height": 2160},
        # the differentiable configuration: 50k vertices, 8 instances, 8 cameras at 512x512
        {"name": "fit_50k_mixed", "kind": "fit", "frequency": 71, "instances": 8, "cameras": 8, "width": 512,
         "height": 512, "precision": "mixed"},
        # a small fit's inner loop: latency and launches
        {"name": "fit_small_f32", "kind": "fit", "frequency": 16, "instances": 1, "cameras": 2, "width": 128,
         "height": 128, "precision": "float32"},
        # a gradient check's precision, odd non-square views
        {"name": "fit_mid_f64", "kind": "fit", "frequency": 40, "instances": 4, "cameras": 3, "width": 401,
         "height": 301, "precision": "float64"},
        # the transform update of a large animated forest
        {"name": "animate_64k", "kind": "animate", "nodes": 65536},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["view", "view", "still", "cut", "player", "views", "pose", "pose", "fit", "fit", "fit", "preview",
                       "animate"])
    if kind == "animate":
        return {"kind": kind, "nodes": _log(rng, 50, 65536)}
    if kind in ("fit", "preview"):
        return {"kind": kind, "frequency": _log(rng, 8, 71), "instances": _log(rng, 1, 8), "cameras": _log(rng, 1, 8),
                "width": _log(rng, 64, 512), "height": _log(rng, 64, 512),
                "precision": rng.choice(["mixed", "mixed", "float32", "float64"])}
    c = {"kind": kind, "scene": "spheres", "objects": _log(rng, 16, 512)}
    if kind == "views":
        return {**c, "views": _log(rng, 2, 16), "mode": rng.choice(["flat", "bary", "bary"])}
    if kind == "pose":
        if rng.random() < 0.3:
            c["scene"], c["objects"] = "uneven", rng.choice([4, 5])
        return {**c, "views": _log(rng, 1, 8), "width": _log(rng, 160, 1280), "height": _log(rng, 120, 720)}
    if kind in ("view", "cut") and rng.random() < 0.4:
        c["scene"], c["objects"] = "city", 0
    small = kind in ("still", "player")
    c["width"], c["height"] = _log(rng, 96, 1280 if small else 3840), _log(rng, 64, 720 if small else 2160)
    if kind != "player":
        c["mode"] = rng.choice(["reference", "flat", "bary", "bary", "cone"])
    if kind == "cut":
        c["frames"] = rng.randint(1, 4)
    return c


# -- scenes and cameras ---------------------------------------------------------
def _scene(case, seed):
    if case["scene"] == "city":
        return Scene(2, seed).arrays()
    if case["scene"] == "uneven":     # one set of meshes, its instances moved by the seed
        sc = _uneven(case["objects"])
        move = np.random.default_rng(seed).normal(0.0, 20.0, (len(sc.transforms), 3)).astype(np.float32)
        move[:, 1] *= 0.1
        xf = sc.transforms.copy()
        xf[:, 12:15] += move
        return dataclasses.replace(sc, transforms=xf)
    return Scene(1, seed, case["objects"]).arrays()


@functools.lru_cache(maxsize=2)
def _uneven(halvings):
    """The uneven stress scene, its 200 meshes halved that many times."""
    return Scene(5, 5, halvings).arrays()


def _street(rng, width, height):
    """A camera in one of the city's streets, looking down it."""
    z = 12.0 * int(rng.integers(-8, 9))
    eye = np.array([-384.0 + 12.0 * rng.uniform(0.3, 8.0), 1.7, z])
    target = eye + np.array([100.0, 0.0, 100.0 * math.tan(math.radians(rng.uniform(-4.0, 4.0)))])
    return view_desc(width, height, eye.tolist(), target.tolist(), fovy_deg=60.0)


def _orbit(rng, width, height, radius):
    a = rng.uniform(0.0, 2.0 * math.pi)
    eye = (radius * math.cos(a), rng.uniform(0.05, 0.35) * radius, radius * math.sin(a))
    return view_desc(width, height, eye, rng.uniform(-10.0, 10.0, 3).tolist(), fovy_deg=rng.uniform(45.0, 75.0))


def _view_desc(case, rng):
    if case["scene"] == "city":
        return _street(rng, case["width"], case["height"])
    return _orbit(rng, case["width"], case["height"], rng.uniform(90.0, 120.0))


def _uneven_sizes(case):
    """View sizes: the first the case's own, the others down to a quarter of it."""
    rng = np.random.default_rng(case["views"])
    out = [(case["width"], case["height"])]
    while len(out) < case["views"]:
        out.append(tuple(max(32, int(s * rng.uniform(0.25, 1.0))) for s in out[0]))
    return out


def _texture(vertices):
    """Planar uvs for a mesh's vertices."""
    v = vertices.copy()
    p = v["position"]
    v["uv"] = np.stack([p[:, 0] * 0.5, p[:, 2] * 0.5 + p[:, 1] * 0.25], 1).astype(np.float16).view(np.uint16)
    return v


# -- animated forests -----------------------------------------------------------
def _forest(nodes, seed, spread=1.0, roots=None):
    """A random forest of mesh nodes, half of them driven by 1 to 3 channels of
    random path and interpolation with 2 to 16 keys.  Returns it with each
    node's parent and its depth-first position (the order of the transforms)."""
    rng = np.random.default_rng(seed)
    roots = min(nodes, roots or max(1, nodes // 64))
    parent = np.full(nodes, -1, np.int64)
    parent[roots:] = (rng.random(nodes - roots) * np.arange(roots, nodes)).astype(np.int64)
    order = np.argsort(parent, kind="stable")
    kids = order[parent[order] >= 0]
    counts = np.bincount(parent[parent >= 0], minlength=nodes)
    first = np.concatenate([[0], np.cumsum(counts)[:-1]])
    nd = np.zeros(nodes, NODE_DTYPE)
    nd["first_child"], nd["child_count"] = first, counts
    nd["translation"] = rng.normal(0.0, spread, (nodes, 3))
    q = rng.normal(size=(nodes, 4))
    nd["rotation"] = q / np.linalg.norm(q, axis=1, keepdims=True)
    nd["scale"] = rng.uniform(0.8, 1.2, (nodes, 3))
    ch_node = np.nonzero(rng.random(nodes) < 0.5)[0]
    ch_node = np.repeat(ch_node, rng.integers(1, 4, len(ch_node)))
    n = len(ch_node)
    path, interp, keys = rng.integers(0, 3, n), rng.integers(0, 3, n), rng.integers(2, 17, n)
    outs, comps = keys * np.where(interp == N.INTERP_CUBICSPLINE, 3, 1), np.where(path == N.PATH_ROTATION, 4, 3)
    t_off = np.concatenate([[0], np.cumsum(keys)[:-1]])[:n]
    v_off = np.concatenate([[0], np.cumsum(outs * comps)[:-1]])[:n]
    seg = np.repeat(np.arange(n), keys)
    times = rng.uniform(0.1, 4.0, int(keys.sum())).astype(np.float32)
    times = times[np.lexsort((times, seg))]
    values = rng.normal(0.0, 1.0, int((outs * comps).sum())).astype(np.float32)
    # animated scales stay positive and near 1, animated translations at the spread
    which = np.repeat(path, outs * comps)
    values = np.where(which == N.PATH_SCALE, np.exp(0.1 * values),
                      np.where(which == N.PATH_TRANSLATION, spread * values, values)).astype(np.float32)
    sp, ch = np.zeros(n, ANIM_SAMPLER_DTYPE), np.zeros(n, ANIM_CHANNEL_DTYPE)
    sp["input_offset"], sp["input_count"], sp["output_offset"], sp["interpolation"] = t_off, keys, v_off, interp
    ch["node"], ch["sampler"], ch["path"] = ch_node, np.arange(n), path
    h = Hierarchy(nd, kids.astype(np.uint32), np.arange(roots, dtype=np.uint32), sp, times, values, ch)
    return h, parent


def _depth_first(h):
    out, stack = [], [int(r) for r in h.roots[::-1]]
    first, count = h.nodes["first_child"], h.nodes["child_count"]
    while stack:
        n = stack.pop()
        out.append(n)
        stack.extend(int(k) for k in h.children[first[n]:first[n] + count[n]][::-1])
    return np.array(out)


# -- differentiable scenes --------------------------------------------------------
def _fit_inputs(case, seed):
    """Positions [V, 3], triangles, albedo [V, 3], transforms, camera matrices
    and the loss gradient of the image, on the GPU."""
    s = D.c4_scene(seed=seed, instances=case["instances"], cameras=case["cameras"], size=64,
                   frequency=case["frequency"])
    W, H = case["width"], case["height"]
    rng = np.random.default_rng(seed)
    vps = []
    for k in range(case["cameras"]):
        a = 2.0 * math.pi * (k + rng.uniform(0.2, 0.8)) / case["cameras"]
        vps.append(D.camera_matrix(view_desc(W, H, (3.0 * math.cos(a), 0.8, 3.0 * math.sin(a)), (0.0, 0.0, 0.0),
                                             fovy_deg=45.0)))
    pos = s.pos + rng.normal(0.0, 0.1 / case["frequency"], s.pos.shape).astype(np.float32)
    g = torch.Generator("cuda").manual_seed(seed)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    g_img = 0.1 * torch.randn((case["cameras"], H, W, 3), generator=g, device="cuda",
                              dtype=torch.float64 if case["precision"] == "float64" else torch.float32)
    return dev(pos), dev(s.tris), dev(s.albedo), dev(s.xforms), dev(np.stack(vps)), g_img


# -- the cases ----------------------------------------------------------------------
def prepare(case, seed):
    kind, rng = case["kind"], np.random.default_rng(seed)
    if kind in ("fit", "preview"):
        pos, tris, alb, xf, vp, g = _fit_inputs(case, seed)
        dt = torch.float64 if case["precision"] == "float64" else torch.float32
        params = [t.to(dt).requires_grad_(kind == "fit") for t in (pos, alb, xf)]
        return {"case": case, "params": params, "tris": tris, "vp": vp, "g": g}
    r = Renderer(0)
    if kind == "animate":
        h, _ = _forest(case["nodes"], seed)
        r.set_hierarchy(h)
        return {"case": case, "r": r, "nodes": case["nodes"], "time": _time_of(seed)}
    sc = _scene(case, seed)
    st = {"case": case, "r": r, "stream": torch.cuda.Stream()}
    if kind == "player":
        sc = dataclasses.replace(sc, meshes=[dataclasses.replace(m, vertices=_texture(m.vertices)) for m in sc.meshes])
        sc.textures = [Texture(rng.integers(0, 256, (256, 256, 4), dtype=np.uint8), k % 3, (k + 1) % 3) for k in range(8)]
        sc.materials = sc.materials.copy()
        sc.materials["albedo_index"] = np.arange(len(sc.materials)) % 8
        h, _ = _forest(len(sc.transforms), seed, spread=25.0, roots=len(sc.transforms) // 4)
        r.load(sc)
        r.set_hierarchy(h)
        vd = _view_desc(case, rng)
        st.update(view=r.create_view(vd.width, vd.height), cam=camera_from_view(vd), time=_time_of(seed))
        return st
    r.load(sc)
    if kind == "views":
        vds = Scene(3, seed).arrays().views
        vds = (vds[0:4:2] + vds[4:10:3] + vds[10:])[:case["views"]]     # cascades, cube faces, cameras
        sizes = np.random.default_rng(3)
        for v in vds[4:]:
            v.width, v.height = int(sizes.integers(256, 1921)), int(sizes.integers(256, 1081))
        views = [r.create_view(v.width, v.height) for v in vds]
        st.update(views=views, cams=[camera_from_view(v) for v in vds], batch=r.create_batch(views),
                  flags=MODES[case["mode"]] | N.GRAPH, out=[_image(v) for v in vds])
        return st
    if kind == "pose":
        radius = 350.0 if case["scene"] == "uneven" else 100.0
        vds = [_orbit(rng, w, h, radius) for w, h in _uneven_sizes(case)]
        views = [r.create_view(v.width, v.height) for v in vds]
        with torch.cuda.stream(st["stream"]):
            g = torch.Generator("cuda").manual_seed(seed)
            st.update(frame=DifferentiableFrame(r, views, [camera_from_view(v) for v in vds]),
                      transforms=torch.from_numpy(sc.transforms).cuda(),
                      g=[torch.randn((v.height, v.width, 3), generator=g, device="cuda") for v in vds])
        return st
    vd = _view_desc(case, rng)
    st.update(view=r.create_view(vd.width, vd.height), cams=[camera_from_view(vd)], flags=MODES[case["mode"]],
              eye=tuple(vd.eye), out=_image(vd))
    if kind == "cut":
        step = 1.5 * (np.array(vd.target) - np.array(vd.eye)) / 100.0
        for _ in range(case["frames"] - 1):
            for k in range(3):
                vd.eye[k] += step[k]
                vd.target[k] += step[k]
            st["cams"].append(camera_advance(st["cams"][-1], vd))
    else:   # a program that already runs: the frames before this one
        for _ in range(2):
            st["view"].render(st["cams"][0], st["flags"], st["eye"])
    r.sync()
    return st


def _image(vd):
    return torch.empty((vd.height, vd.width, 3), dtype=torch.float32, device="cuda")


def _time_of(seed):
    return 0.5 + (seed % 1013) * 0.00731


def run(state):
    kind = state["case"]["kind"]
    if kind in ("fit", "preview"):
        c = state["case"]
        pos, alb, xf = state["params"]
        img, ids, _ = D.render(pos, alb, state["tris"], xf, state["vp"], c["height"], c["width"],
                               precision=c["precision"])
        if kind == "preview":
            return {"image": img, "ids": ids}
        g = torch.autograd.grad(img, state["params"], state["g"])
        return {"image": img.detach(), "ids": ids, "g_positions": g[0], "g_albedo": g[1], "g_transforms": g[2]}
    r = state["r"]
    if kind == "animate":
        r.update_transforms(state["time"])
        return {"transforms": r.read_transforms(state["nodes"])}
    if kind == "still":
        state["view"].render(state["cams"][0], state["flags"], state["eye"])
        return {"color": state["view"].color()}
    if kind == "player":
        r.update_transforms(state["time"])
        state["time"] += 1.0 / 60.0
        state["view"].render(state["cam"], TWO_PASS | N.RESOLVE_TEXTURED | N.MOTION_VECTORS)
        return {"color": state["view"].color(), "motion": state["view"].motion()}
    stream = state["stream"]
    with torch.cuda.stream(stream):
        if kind == "views":
            state["batch"].render(state["cams"], state["flags"], stream=stream.cuda_stream)
            return {"images": [v.aa_image(c, o) for v, c, o in zip(state["views"], state["cams"], state["out"])]}
        if kind == "pose":
            t = state["transforms"].detach().requires_grad_()
            images = state["frame"](t)
            (g,) = torch.autograd.grad(images, t, state["g"])
            return {"images": [i.detach() for i in images], "g_transforms": g}
        if kind == "cut":
            state["view"].reset_history()
        for cam in state["cams"]:
            state["view"].render(cam, state["flags"], state["eye"], stream=stream.cuda_stream)
        return {"image": state["view"].aa_image(state["cams"][-1], state["out"])}


def work(case):
    """Bytes of the inputs read once and the outputs written once; operations
    of the arithmetic that the outputs need."""
    kind = case["kind"]
    if kind == "animate":   # per node: 40 B TRS, 64 B matrix, half of them 2 channels of about 9 keys; 3 products a node
        return {"bytes": case["nodes"] * (40 + 64 + 2 * (16 + 9 * 4 + 24)), "flops": case["nodes"] * 3 * 112}
    if kind in ("fit", "preview"):
        V, T = 10 * case["frequency"] ** 2 + 2, 20 * case["frequency"] ** 2
        ci, px = case["cameras"] * case["instances"], case["cameras"] * case["width"] * case["height"]
        e = 8 if case["precision"] == "float64" else 4
        both = 2 if kind == "fit" else 1
        # image (and its gradient), ids, positions, albedo and gradients; a vertex transform is 28 operations, a
        # triangle's setup about 60, a pixel's interpolation about 60 (twice that again for the gradients)
        return {"bytes": px * (3 * e * both + 4) + V * 6 * e * both + T * 12,
                "flops": ci * (28 * V + 60 * T) + px * 60 * (3 if kind == "fit" else 1)}
    meshlets = 62           # of a 5120-triangle sphere
    if case["scene"] == "city":
        draws, transforms = 126976, 6144
    elif case["scene"] == "uneven":
        draws, transforms = 15_200_000 >> case["objects"], 6900 >> case["objects"]
    else:
        draws, transforms = meshlets * case["objects"], case["objects"]
    frames = case.get("frames", 1)
    if kind == "views":     # half the views up to 2048^2, the rest about 1 Mpx
        px = case["views"] * 850_000
    else:
        px = case["width"] * case["height"] * (1 + 0.4 * (case.get("views", 1) - 1))
    # a draw's record and bounds, a transform, and per pixel the colour, the linear image or read-back colour (and its
    # gradient for a pose, and the motion vector for a player)
    out = 4 + {"still": 4, "player": 12, "pose": 24}.get(kind, 12)
    return {"bytes": frames * (36 * draws + 64 * transforms + 12 * px) + out * px,
            "flops": frames * case.get("views", 1) * 60 * draws + frames * 60 * px}


# -- 64-bit values ------------------------------------------------------------------
def exact(case, seed):
    if case["kind"] == "animate":
        return {"transforms": _exact_transforms(*_forest(case["nodes"], seed), _time_of(seed))}
    if case["kind"] not in ("fit", "preview"):
        return None
    pos, tris, alb, xf, vp, g = _fit_inputs(case, seed)
    fit = case["kind"] == "fit"
    pos, alb, xf = (t.double().requires_grad_(fit) for t in (pos, alb, xf))
    A = torch.matmul(vp.double()[:, None], xf[None])                                   # [C, I, 4, 4]
    hom = torch.cat([pos, torch.ones_like(pos[:, :1])], 1)
    clip = torch.matmul(hom[None, None], A.transpose(-1, -2).contiguous())             # [C, I, V, 4]
    depth, ids = _exact_raster(clip.detach().float(), tris.long(), case["height"], case["width"])
    img = _exact_shade(clip, alb, tris.long(), ids, depth)
    if not fit:
        return {"image": img, "ids": None}
    grads = torch.autograd.grad(img, (pos, alb, xf), g.double())
    return {"image": img.detach(), "ids": None, "g_positions": grads[0], "g_albedo": grads[1], "g_transforms": grads[2]}


def _exact_raster(clip, tris, H, W):
    """Depth [C, H, W] and ids (0, or instance * T + triangle + 1): vertices
    snapped to 1/256 pixel, integer edge functions with a top-left rule, the
    depth plane's value at the centres, the nearest triangle."""
    C, I, V, _ = clip.shape
    T = len(tris)
    half = torch.tensor([W * 0.5, H * 0.5], device=clip.device)
    snap = torch.round((half * (clip[..., :2] / clip[..., 3:]) + half) * 256.0).long()
    z = clip[..., 2] / clip[..., 3]
    keys = torch.full((C * H * W,), -1, dtype=torch.int64, device=clip.device)
    for c in range(C):
        P, Z = snap[c][:, tris].reshape(I * T, 3, 2), z[c][:, tris].reshape(I * T, 3)
        cross = lambda a, b: a[:, 0] * b[:, 1] - a[:, 1] * b[:, 0]
        area = cross(P[:, 1] - P[:, 0], P[:, 2] - P[:, 0])
        flip = area < 0
        P, Z = torch.where(flip[:, None, None], P[:, [0, 2, 1]], P), torch.where(flip[:, None], Z[:, [0, 2, 1]], Z)
        lo = torch.clamp((P.amin(1) + 127) >> 8, min=0)
        hi = torch.minimum((P.amax(1) - 128) >> 8, torch.tensor([W - 1, H - 1], device=P.device))
        size = torch.clamp(hi - lo + 1, min=0)
        n = torch.where(area != 0, size[:, 0] * size[:, 1], 0)
        tri = torch.repeat_interleave(torch.arange(I * T, device=P.device), n)
        k = torch.arange(len(tri), device=P.device) - torch.repeat_interleave(torch.cumsum(n, 0) - n, n)
        w = size[tri, 0]
        px = torch.stack([lo[tri, 0] + k % w, lo[tri, 1] + k // w], 1)
        centre = px * 256 + 128
        inside = torch.ones_like(tri, dtype=torch.bool)
        for a, b in ((1, 2), (2, 0), (0, 1)):
            e = P[tri, b] - P[tri, a]
            v = cross(e, centre - P[tri, a])
            inside &= (v > 0) | ((v == 0) & ((e[:, 1] < 0) | ((e[:, 1] == 0) & (e[:, 0] > 0))))
        tri, px, centre = tri[inside], px[inside], centre[inside]
        e1, e2 = (P[:, 1] - P[:, 0]).double() / 256.0, (P[:, 2] - P[:, 0]).double() / 256.0
        d1, d2 = (Z[:, 1].double() - Z[:, 0].double()), (Z[:, 2].double() - Z[:, 0].double())
        det = area.abs().double() / 65536.0
        za, zb = ((d1 * e2[:, 1] - d2 * e1[:, 1]) / det).float(), ((d2 * e1[:, 0] - d1 * e2[:, 0]) / det).float()
        off = (centre - P[tri, 0]).float() * 0.00390625
        zz = Z[tri, 0] + (za[tri] * off[:, 0] + zb[tri] * off[:, 1])
        ok = (zz >= 0.0) & (zz <= 1.0)
        key = (((~((zz[ok] + 0.0).view(torch.int32).long())) & 0xFFFFFFFF) << 32) | (0xFFFFFFFE - (tri[ok] + 1))
        at = (c * H + px[ok, 1]) * W + px[ok, 0]
        keys.scatter_reduce_(0, at, key, "amin")
    empty = keys == -1
    ids = torch.where(empty, 0, 0xFFFFFFFE - (keys & 0xFFFFFFFF))
    depth = torch.where(empty, 0, ~(keys >> 32) & 0xFFFFFFFF).to(torch.int32).view(torch.float32)
    return depth.reshape(C, H, W), ids.reshape(C, H, W)


def _exact_shade(clip, attr, tris, ids, depth):
    """Perspective-correct interpolation, then the analytic edge antialiasing."""
    C, H, W = ids.shape
    T, A = len(tris), attr.shape[1]
    flat = ids.reshape(-1)
    dev = clip.device

    def corners(p, id_):     # clip positions [n, 3, 4] and vertices of the triangles at pixels p
        v = tris[(id_ - 1) % T]
        return clip[(p // (H * W))[:, None], ((id_ - 1) // T)[:, None], v], v

    def ndc(p):
        return ((p % W).double() + 0.5) / (W * 0.5) - 1.0, ((p // W % H).double() + 0.5) / (H * 0.5) - 1.0

    p = torch.nonzero(flat > 0)[:, 0]
    P, v = corners(p, flat[p])
    xn, yn = ndc(p)
    u = torch.stack([P[..., 0] - xn[:, None] * P[..., 3], P[..., 1] - yn[:, None] * P[..., 3]], -1)
    cross = lambda a, b: a[..., 0] * b[..., 1] - a[..., 1] * b[..., 0]
    l = torch.stack([cross(u[:, 1], u[:, 2]), cross(u[:, 2], u[:, 0]), cross(u[:, 0], u[:, 1])], 1)
    lam = l / l.sum(1, keepdim=True)
    color = torch.zeros((C * H * W, A), dtype=torch.float64, device=dev).index_put((p,), (lam[..., None] * attr[v]).sum(1))
    out = color
    pix = torch.arange(C * H * W, device=dev).reshape(C, H, W)
    for dx, dy in ((1, 0), (0, 1)):
        a, b = pix[:, :H - dy, :W - dx].reshape(-1), pix[:, dy:, dx:].reshape(-1)
        differ = flat[a] != flat[b]
        a, b = a[differ], b[differ]
        za, zb = depth.reshape(-1)[a], depth.reshape(-1)[b]
        a_front = torch.where(flat[a] == 0, False, torch.where(flat[b] == 0, True, za >= zb))
        f, k = torch.where(a_front, a, b), torch.where(a_front, b, a)
        P, _ = corners(f, flat[f])
        xc, yc = ndc(f)
        S = torch.stack([W * 0.5 * (P[..., 0] / P[..., 3] - xc[:, None]),
                         H * 0.5 * (P[..., 1] / P[..., 3] - yc[:, None])], -1)
        step = torch.where(a_front, 1.0, -1.0).double()
        cb = torch.stack([step * dx, step * dy], -1)
        sgn = torch.sign(cross(S[:, 1] - S[:, 0], S[:, 2] - S[:, 0])).detach()
        edge = S[:, [1, 2, 0]] - S
        ef = sgn[:, None] * cross(edge, -S)
        eb = sgn[:, None] * cross(edge, cb[:, None] - S)
        ok = (ef >= 0) & (eb <= 0) & (ef > eb)
        t = torch.where(ok, ef / torch.where(ok, ef - eb, 1.0), 2.0)
        first = t.argmin(1)
        hit = ok.any(1) & (sgn != 0)
        t = t.gather(1, first[:, None])[:, 0][hit]
        f, k = f[hit], k[hit]
        to_front = t < 0.5
        tgt, src = torch.where(to_front, f, k), torch.where(to_front, k, f)
        alpha = torch.where(to_front, 0.5 - t, t - 0.5)
        out = out.index_add(0, tgt, alpha[:, None] * (color[src] - color[tgt]))
    return out.reshape(C, H, W, A)


def _exact_transforms(h, parent, time):
    """The animated TRS of every node and the product down its ancestors."""
    nd = h.nodes
    trs = [nd["translation"].astype(np.float64), nd["rotation"].astype(np.float64), nd["scale"].astype(np.float64)]
    time = np.float32(time)
    for ch in h.channels:
        s = h.samplers[ch["sampler"]]
        key = h.times[s["input_offset"]:s["input_offset"] + s["input_count"]].astype(np.float64)
        width, cubic = (4 if ch["path"] == N.PATH_ROTATION else 3), s["interpolation"] == N.INTERP_CUBICSPLINE
        n = len(key) * (3 if cubic else 1)
        val = h.values[s["output_offset"]:s["output_offset"] + n * width].astype(np.float64).reshape(n, width)
        if cubic:
            tin, val, tout = val[0::3], val[1::3], val[2::3]
        x = math.fmod(float(time), key[-1])
        i = int(np.searchsorted(key, x, side="left"))
        if i == 0 or i == len(key):
            o = val[0 if i == 0 else -1]
        else:
            dt = key[i] - key[i - 1]
            t = (x - key[i - 1]) / dt
            a, b = val[i - 1], val[i]
            if s["interpolation"] == N.INTERP_STEP:
                o = a
            elif cubic:
                o = (a * (2 * t ** 3 - 3 * t ** 2 + 1) + tout[i - 1] * dt * (t ** 3 - 2 * t ** 2 + t)
                     + b * (-2 * t ** 3 + 3 * t ** 2) + tin[i] * dt * (t ** 3 - t ** 2))
                if width == 4:
                    o = o / np.linalg.norm(o)
            elif width == 3:
                o = a * (1 - t) + b * t
            else:
                cosv = a @ b
                b, cosv = (-b, -cosv) if cosv < 0 else (b, cosv)
                if cosv > 1.0 - 1.1920928955078125e-7:
                    o = a * (1 - t) + b * t
                else:
                    ang = math.acos(min(cosv, 1.0))
                    o = (math.sin((1 - t) * ang) * a + math.sin(t * ang) * b) / math.sin(ang)
        trs[{N.PATH_TRANSLATION: 0, N.PATH_ROTATION: 1, N.PATH_SCALE: 2}[int(ch["path"])]][ch["node"]] = o
    t, (x, y, z, w), s = trs[0], trs[1].T, trs[2]
    one = np.ones_like(x)
    R = np.stack([np.stack([one - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y)], -1),
                  np.stack([2 * (x * y + w * z), one - 2 * (x * x + z * z), 2 * (y * z - w * x)], -1),
                  np.stack([2 * (x * z - w * y), 2 * (y * z + w * x), one - 2 * (x * x + y * y)], -1)], -2)
    local = np.zeros((len(nd), 4, 4))
    local[:, :3, :3] = R * s[:, None, :]
    local[:, :3, 3], local[:, 3, 3] = t, 1.0
    world, done = local.copy(), parent < 0
    while not done.all():
        now = ~done & (done[np.maximum(parent, 0)])
        world[now] = world[parent[now]] @ local[now]
        done |= now
    return world.transpose(0, 2, 1).reshape(-1, 16)[_depth_first(h)]
