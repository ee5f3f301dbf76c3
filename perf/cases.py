"""The work this framework is measured on: octree raymarching and octree
construction through the public entry points, from one launch of a thousand
rays to 8192^3 terrain at 4K and 2048^3 builds of two million triangles.

A case is a dict of plain values. "kind" picks the entry point:

  rays     raymarch_batch_device: rays a program holds itself (picking,
           collision and visibility queries)
  primary  render_primary_device, or a TilePlan kept for the image size
  batch    Renderer.render_device: many views of one or many octrees per call
  frame    render_frame_device: the viewer's shaded frame
  shadow   render_shadow_device: primary and hard-shadow rays
  build    build_from_mesh / build_from_grid / build_from_terrain, then upload
  oct      encode, from_bytes, upload: the .oct file in both directions

"scene" and "res" name the octree: "grid" a dense volume of spheres and tori
(the solid shell of a signed-distance scene), "mesh" a displaced sphere of
about 20 * (316 * res / 2048)^2 triangles, "terrain" an fBm heightfield.
"""
import math

import numpy as np
import torch

from __graft_entry__ import _import_package

pkg = _import_package()

THREADS = 8          # the builder's sub-block partition
BUDGET = 1 << 30     # the builder's memory budget
LIGHT_EPS = 0.25     # shadow ray pull-back, in voxels


def listed():
    return [
        # a pick or a collision query: a handful of rays against a small octree, launch latency
        {"name": "rays_1k_grid256", "kind": "rays", "scene": "grid", "res": 256, "n": 1021, "lod": False},
        # bulk incoherent rays with a level-of-detail cut-off per ray (visibility or sound queries)
        {"name": "rays_1m_lod_mesh1024", "kind": "rays", "scene": "mesh", "res": 1024, "n": 1000003, "lod": True},
        # one 720p image of a 256^3 scene, a single call with nothing kept between calls
        {"name": "primary_720p_grid256", "kind": "primary", "scene": "grid", "res": 256, "width": 1280, "height": 720,
         "plan": False},
        # one 1080p view of the 2048^3 mesh octree, rendered again and again through a tile plan
        {"name": "primary_1080p_plan_mesh2048", "kind": "primary", "scene": "mesh", "res": 2048, "width": 1920,
         "height": 1080, "plan": True},
        # eight 1080p views of one 2048^3 octree in one launch (an offline or multi-user render)
        {"name": "batch_8x1080p_mesh2048", "kind": "batch", "scene": "mesh", "res": 2048, "trees": 1, "views": 8,
         "width": 1920, "height": 1080, "mixed": False},
        # a render service's launch: many octrees of different sizes, views of mixed odd sizes
        {"name": "batch_16trees_64views", "kind": "batch", "scene": "mixed", "res": 1024, "trees": 16, "views": 64,
         "width": 1920, "height": 1080, "mixed": True},
        # the viewer's frame (coarse pass, fine pass, shading) as consecutive frames run it
        {"name": "frame_1080p_plan_mesh2048", "kind": "frame", "scene": "mesh", "res": 2048, "width": 1920,
         "height": 1080, "stride": 1, "plan": True},
        # a 4K image of an 8192^3 terrain with hard shadows: the deepest octree and the largest image
        {"name": "shadow_4k_plan_terrain8192", "kind": "shadow", "scene": "terrain", "res": 8192, "width": 3840,
         "height": 2160, "plan": True},
        # two million triangles to a 2048^3 octree
        {"name": "build_mesh2048", "kind": "build", "scene": "mesh", "res": 2048},
        # an interactive edit: a small mesh voxelized again, bound by launches and round trips
        {"name": "build_mesh256", "kind": "build", "scene": "mesh", "res": 256},
        # a raw volume of odd sizes (a scan) to an octree
        {"name": "build_grid_odd", "kind": "build", "scene": "grid", "res": 256, "width": 203, "height": 251,
         "depth": 189},
        # an octree saved to and loaded from an .oct image
        {"name": "oct_roundtrip_mesh512", "kind": "oct", "scene": "mesh", "res": 512},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["rays", "primary", "primary", "batch", "batch", "frame", "shadow", "build", "build", "oct"])
    if kind == "oct":
        return {"kind": kind, "scene": "mesh", "res": _log_int(rng, 64, 512)}
    if kind == "build":
        scene = rng.choice(["mesh", "mesh", "grid", "terrain"])
        if scene == "mesh":
            return {"kind": kind, "scene": scene, "res": _log_int(rng, 64, 2048)}
        if scene == "terrain":
            return {"kind": kind, "scene": scene, "res": 1 << rng.randint(7, 12)}
        return {"kind": kind, "scene": scene, "res": 256, "width": _log_int(rng, 24, 256),
                "height": _log_int(rng, 24, 256), "depth": _log_int(rng, 24, 256)}
    scene = rng.choice(["grid", "mesh", "mesh", "terrain"])
    if scene == "grid":
        res = 1 << rng.randint(6, 8)
    elif scene == "mesh":
        res = _log_int(rng, 128, 2048)
    else:
        res = 1 << rng.randint(9, 13)
    case = {"kind": kind, "scene": scene, "res": res}
    if kind == "rays":
        case.update(n=_log_int(rng, 64, 1000000), lod=rng.random() < 0.5)
        return case
    width = _log_int(rng, 160, 1920)
    case.update(width=width, height=max(90, int(width / rng.choice([4 / 3, 16 / 9, 1.0]) + rng.randint(-3, 3))))
    if kind == "batch":
        case.update(trees=rng.randint(1, 8), views=_log_int(rng, 2, 32), mixed=rng.random() < 0.5)
        if case["mixed"]:
            case.update(scene="mixed", res=512)
        elif scene == "terrain":
            case.update(res=min(res, 2048))
    else:
        case["plan"] = rng.random() < 0.5
        if kind == "frame":
            case["height"] = (case["height"] + 15) // 16 * 16  # the viewer's 16 stripes, none empty
            case["stride"] = rng.choice([1, 1, 3])
    return case


# ---- scenes -----------------------------------------------------------------


def _primitives(seed):
    """16 spheres and tori: centres U[0,1]^3, radii U[0.05,0.2]."""
    rng = np.random.default_rng(seed)
    prims = []
    for _ in range(16):
        axis = rng.normal(size=3)
        r1, r2 = rng.uniform(0.05, 0.2, 2)
        prims.append((int(rng.integers(0, 2)), rng.uniform(0.0, 1.0, 3).tolist(), float(r1), float(min(r1, r2)),
                      (axis / np.linalg.norm(axis)).tolist()))
    return prims


def _sdf(prims, x, y, z):
    d = torch.full_like(x, 10.0)
    for kind, c, r1, r2, a in prims:
        qx, qy, qz = x - c[0], y - c[1], z - c[2]
        qq = qx * qx + qy * qy + qz * qz
        if kind == 0:
            di = qq.sqrt() - r1
        else:
            h = qx * a[0] + qy * a[1] + qz * a[2]
            rad = (qq - h * h).clamp_min(0.0).sqrt() - r1
            di = (rad * rad + h * h).sqrt() - r2
        d = torch.minimum(d, di)
    return d


def _volume(seed, n, w, h, d):
    """uint32 words (as int64 on the device, [d, h, w]) of the scene's shell: 0
    where empty, elsewhere the surface normal and a shade packed as a leaf word
    (sign, dominant axis, two 11-bit quotients, 7-bit shade)."""
    prims = _primitives(seed)
    out = torch.zeros(d, h, w, dtype=torch.int64, device="cuda")
    ax = [(torch.arange(k, device="cuda", dtype=torch.float64) + 0.5) / n for k in (w, h, d)]
    for z0 in range(0, d, 64):
        z, y, x = torch.meshgrid(ax[2][z0:z0 + 64], ax[1], ax[0], indexing="ij")
        at = (_sdf(prims, x, y, z).abs() <= 0.5 * math.sqrt(3.0) / n).nonzero(as_tuple=True)
        x, y, z = x[at], y[at], z[at]
        e = 1.0 / n
        g = torch.stack([_sdf(prims, x + e, y, z) - _sdf(prims, x - e, y, z),
                         _sdf(prims, x, y + e, z) - _sdf(prims, x, y - e, z),
                         _sdf(prims, x, y, z + e) - _sdf(prims, x, y, z - e)])
        dom, face = g.abs().max(0)
        dom = dom.clamp_min(1e-12)
        sign = (g.gather(0, face[None])[0] < 0).long()
        n1 = g.gather(0, torch.where(face == 2, 0, face + 1)[None])[0] / dom
        n2 = g.gather(0, torch.where(face == 0, 2, face - 1)[None])[0] / dom
        u = ((n1 * 0.5 + 0.5) * 2047.0).long().clamp(0, 2047)
        v = ((n2 * 0.5 + 0.5) * 2047.0).long().clamp(0, 2047)
        out[at[0] + z0, at[1], at[2]] = (sign << 31) | (face << 29) | (u << 18) | (v << 7) | 101
    return out


def _grid(seed, n, w, h, d):
    return _volume(seed, n, w, h, d).cpu().numpy().astype(np.uint32)


def _mesh(seed, res):
    """A cube-sphere displaced by six octaves of sine noise (5% of the radius):
    the vertex table and faces of build_from_mesh."""
    k = max(2, round(408 * res / 2048))
    g = torch.Generator().manual_seed(seed)
    lin = torch.linspace(-1.0, 1.0, k + 1, dtype=torch.float64, device="cuda")
    a, b = torch.meshgrid(lin, lin, indexing="ij")
    a, b, one = a.reshape(-1), b.reshape(-1), torch.ones((k + 1) ** 2, dtype=torch.float64, device="cuda")
    p = torch.cat([torch.stack(f, 1) for f in ((one, a, b), (-one, b, a), (b, one, a), (a, -one, b), (a, b, one),
                                               (b, a, -one))])
    p = p / p.norm(dim=1, keepdim=True)
    r, amp, freq = torch.ones(len(p), dtype=torch.float64, device="cuda"), 0.5, 4.0
    for _ in range(6):
        m = torch.randn(3, 3, generator=g, dtype=torch.float64).cuda()
        ph = (torch.rand(3, generator=g, dtype=torch.float64) * 6.28318).cuda()
        r = r + 0.05 * amp * torch.sin(freq * (p[:, :1] * m[0] + p[:, 1:2] * m[1] + p[:, 2:] * m[2]) + ph).prod(1)
        amp, freq = amp * 0.5, freq * 2.0
    p = p * r[:, None]
    i, j = torch.meshgrid(torch.arange(k, device="cuda"), torch.arange(k, device="cuda"), indexing="ij")
    q = (i * (k + 1) + j).reshape(-1)
    quad = torch.stack([q, q + k + 1, q + k + 2, q, q + k + 2, q + 1], 1).reshape(-1, 3)
    faces = (quad[None] + (torch.arange(6, device="cuda") * (k + 1) ** 2)[:, None, None]).reshape(-1, 3)
    table = torch.zeros(len(p), 9, dtype=torch.float32, device="cuda")
    table[:, :3] = p.float()
    table[:, 6:] = 255.0
    return table.cpu().numpy(), np.full(len(faces), 3, np.int32), faces.reshape(-1).int().cpu().numpy()


def _tree(scene, res, seed):
    if scene == "terrain":
        return pkg.VoxelOctree.build_from_terrain(res, seed, memory_budget=BUDGET)
    if scene == "grid":
        return pkg.VoxelOctree.build_from_grid(_grid(seed, res, res, res, res), memory_budget=BUDGET)
    table, counts, idx = _mesh(seed, res)
    return pkg.VoxelOctree.build_from_mesh(table, False, counts, idx, res, threads=THREADS, memory_budget=BUDGET)


# ---- cameras and rays ---------------------------------------------------------


def _camera(rng, scene):
    """An orbit camera around the unit cube at [1,2]^3: the 16 floats of its
    transform (columns right, up, forward, translation) and its position. The
    terrain is seen from above at radius 1; the other scenes from U[0.9,1.4]."""
    yaw = rng.uniform(0.0, 2.0 * math.pi)
    pitch = rng.uniform(0.4, 0.9) if scene == "terrain" else rng.uniform(-1.0, 1.0)
    radius = 1.0 if scene == "terrain" else rng.uniform(0.9, 1.4)
    fwd = np.array([math.cos(pitch) * math.sin(yaw), -math.sin(pitch), math.cos(pitch) * math.cos(yaw)])
    right = np.array([math.cos(yaw), 0.0, -math.sin(yaw)])
    up = np.cross(fwd, right)
    m = np.zeros((4, 4), np.float32)
    m[:3, 0], m[:3, 1], m[:3, 2], m[:3, 3], m[3, 3] = right, up, fwd, -radius * fwd, 1.0
    return m, (1.5 - radius * fwd).astype(np.float32)


def _svo_camera(m, pos):
    cam = pkg.svo.Camera()
    cam.tform[:] = m.reshape(-1).tolist()
    cam.pos[:] = pos.tolist()
    return cam


def _query_rays(case, seed):
    """Rays from around and inside the cube toward points of its middle."""
    g = torch.Generator().manual_seed(seed + 7)
    n = case["n"]
    o = 1.5 + (torch.rand(n, 3, generator=g) - 0.5) * 1.6
    d = 1.5 + (torch.rand(n, 3, generator=g) - 0.5) * 0.8 - o
    d = d / d.norm(dim=1, keepdim=True).clamp_min(1e-6)
    rs = torch.rand(n, generator=g) * (8.0 / case["res"]) if case["lod"] else None
    return o.cuda(), d.cuda(), None if rs is None else rs.cuda()


def _light(rng):
    el, az = math.radians(rng.uniform(20.0, 60.0)), rng.uniform(0.0, 2.0 * math.pi)
    return np.array([math.cos(el) * math.cos(az), math.sin(el), math.cos(el) * math.sin(az)], np.float32)


def _ray_outputs(n):
    return {"hit": torch.zeros(n, dtype=torch.uint8, device="cuda"),
            "normal": torch.zeros(n, dtype=torch.int32, device="cuda"),
            "t": torch.zeros(n, dtype=torch.float32, device="cuda"),
            "leaf": torch.zeros(n, dtype=torch.int64, device="cuda")}


def _mixed_trees(case, seed):
    rng = np.random.default_rng(seed + 11)
    return [(("mesh", "grid")[i % 2], int(case["res"] >> int(rng.integers(0, 4)))) for i in range(case["trees"])]


def _view_sizes(case):
    if not case["mixed"]:
        return [(case["width"], case["height"])] * case["views"]
    rng = np.random.default_rng(case["views"])
    out = []
    for _ in range(case["views"]):
        w = int(round(math.exp(rng.uniform(math.log(min(320, case["width"])), math.log(case["width"])))))
        out.append((w, max(8, int(round(w / (4 / 3 if rng.random() < 0.5 else 16 / 9))))))
    return out


# ---- the contract -------------------------------------------------------------


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed + 3)
    s = {"case": case, "kind": kind}
    if kind == "build":
        if case["scene"] == "mesh":
            s["mesh"] = _mesh(seed, case["res"])
        elif case["scene"] == "grid":
            s["grid"] = _grid(seed, case["res"], case["width"], case["height"], case["depth"])
        else:
            s["seed"] = seed
        s["words"] = torch.zeros(_word_capacity(case), dtype=torch.int32, device="cuda")
        return s
    if kind == "batch":
        specs = _mixed_trees(case, seed) if case["mixed"] else [(case["scene"], case["res"])] * case["trees"]
        s["trees"] = [_tree(sc, min(r, 256) if sc == "grid" else r, seed + 17 * i) for i, (sc, r) in enumerate(specs)]
        sizes = _view_sizes(case)
        s["renderer"] = pkg.svo.Renderer(len(sizes))
        s["out"], s["views"], first = _ray_outputs(sum(w * h for w, h in sizes)), [], 0
        for i, (w, h) in enumerate(sizes):  # the views' images one after another in each array
            tree = s["trees"][i % len(s["trees"])]
            ptr = {k: v.data_ptr() + first * v.element_size() for k, v in s["out"].items()}
            s["views"].append(pkg.svo.Renderer.view(tree, _svo_camera(*_camera(rng, case["scene"])), w, h, **ptr))
            first += w * h
        for t in s["trees"]:
            t.upload()
        return s
    s["tree"] = _tree(case["scene"], case["res"], seed)
    if kind == "oct":
        s["words"] = torch.zeros(_word_capacity(case), dtype=torch.int32, device="cuda")
        s["file"] = np.zeros(4 * _word_capacity(case), np.uint8)
        return s
    s["tree"].upload()
    if kind == "rays":
        s["rays"] = _query_rays(case, seed)
        s["out"] = _ray_outputs(case["n"])
        return s
    w, h = case["width"], case["height"]
    s["cam"] = _svo_camera(*_camera(rng, case["scene"]))
    if kind == "frame":
        s["plan"] = pkg.svo.TilePlan.for_frame(w, h) if case["plan"] else None
        s["out"] = {"rgba": torch.zeros(w * h, dtype=torch.int32, device="cuda"),
                    "depth": torch.zeros(pkg.svo.frame_depth_count(w, h), dtype=torch.float32, device="cuda")}
        return s
    s["plan"] = pkg.svo.TilePlan(w, h) if case["plan"] else None
    s["out"] = _ray_outputs(w * h)
    if kind == "shadow":
        s["light"] = _light(rng)
        s["out"]["shadow"] = torch.zeros(w * h, dtype=torch.uint8, device="cuda")
    return s


class _DeviceWords:
    """An octree's device words as torch reads foreign device memory."""

    def __init__(self, tree):
        self.__cuda_array_interface__ = {"shape": (tree.word_count(),), "typestr": "<i4", "version": 3,
                                         "data": (tree.upload(), False)}


def _word_capacity(case):
    """Words an octree of the case's kind stays below."""
    if "depth" in case:
        return case["width"] * case["height"] * case["depth"] + 4096
    return {"mesh": 10, "terrain": 4}[case["scene"]] * case["res"] ** 2 + 4096


def _resident_words(tree, words):
    """Copies the words a render reads to the front of `words` (the rest stays 0)."""
    words[:tree.word_count()] = torch.as_tensor(_DeviceWords(tree), device="cuda")
    return words


def run(state):
    kind, case = state["kind"], state["case"]
    stream = torch.cuda.current_stream().cuda_stream
    if kind == "build":
        if case["scene"] == "mesh":
            table, counts, idx = state["mesh"]
            tree = pkg.VoxelOctree.build_from_mesh(table, False, counts, idx, case["res"], threads=THREADS,
                                                   memory_budget=BUDGET)
        elif case["scene"] == "grid":
            tree = pkg.VoxelOctree.build_from_grid(state["grid"], memory_budget=BUDGET)
        else:
            tree = pkg.VoxelOctree.build_from_terrain(case["res"], state["seed"], memory_budget=BUDGET)
        state["tree"] = tree
        return {"words": _resident_words(tree, state["words"]), "count": tree.word_count(), "center": tree.center()}
    if kind == "oct":
        data = state["tree"].encode()
        state["loaded"] = pkg.VoxelOctree.from_bytes(data)
        state["file"][:len(data)] = np.frombuffer(data, np.uint8)
        return {"file": state["file"], "size": len(data), "words": _resident_words(state["loaded"], state["words"])}
    if kind == "batch":
        state["renderer"].render_device(state["views"], stream=stream)
        return state["out"]
    tree, out = state["tree"], state["out"]
    if kind == "rays":
        o, d, rs = state["rays"]
        tree.raymarch_batch_device(case["n"], o.data_ptr(), d.data_ptr(), None if rs is None else rs.data_ptr(), 0.0,
                                   out["hit"].data_ptr(), out["normal"].data_ptr(), out["t"].data_ptr(),
                                   out["leaf"].data_ptr(), stream)
        return out
    w, h, plan = case["width"], case["height"], state["plan"]
    if kind == "frame":
        tree.render_frame_device(state["cam"], w, h, out["rgba"].data_ptr(), out["depth"].data_ptr(),
                                 stride=case["stride"], stream=stream, plan=plan)
    elif kind == "shadow":
        tree.render_shadow_device(state["cam"], w, h, state["light"], LIGHT_EPS / case["res"], out["hit"].data_ptr(),
                                  out["t"].data_ptr(), out["shadow"].data_ptr(), out["normal"].data_ptr(),
                                  out["leaf"].data_ptr(), stream, plan=plan)
    elif plan is not None:
        plan.render_device(tree, state["cam"], out["hit"].data_ptr(), out["normal"].data_ptr(), out["t"].data_ptr(),
                           out["leaf"].data_ptr(), stream)
    else:
        tree.render_primary_device(state["cam"], w, h, out["hit"].data_ptr(), out["normal"].data_ptr(),
                                   out["t"].data_ptr(), out["leaf"].data_ptr(), stream)
    return out


def _octree_words(scene, res):
    """About how many words the scene's octree has (measured shells per res^2)."""
    return int({"mesh": 6.2, "terrain": 2.1, "grid": 5.0}[scene] * res * res)


def work(case):
    kind, depth = case["kind"], max(1, math.ceil(math.log2(case["res"])))
    if kind == "build":
        words = _octree_words(case["scene"], case["res"])
        if case["scene"] == "mesh":
            k = max(2, round(408 * case["res"] / 2048))
            # vertices and faces in, words out; a triangle-box test of ~100 operations per candidate voxel
            return {"bytes": 36 * 6 * (k + 1) ** 2 + 16 * 12 * k * k + 4 * words, "flops": 930 * case["res"] ** 2}
        if case["scene"] == "grid":
            voxels = case["width"] * case["height"] * case["depth"]
            return {"bytes": 4 * voxels + 4 * words, "flops": voxels}
        # eight octaves of value noise per column
        return {"bytes": 4 * words, "flops": 400 * case["res"] ** 2}
    if kind == "oct":
        words = _octree_words(case["scene"], case["res"])
        return {"bytes": 4 * (2 * words) + 2 * 3 * words, "flops": words}
    # a ray visits one node per level at least, with about 20 operations each
    if kind == "rays":
        return {"bytes": case["n"] * (24 + (4 if case["lod"] else 0) + 17), "flops": 20 * depth * case["n"]}
    if kind == "batch":
        rays = sum(w * h for w, h in _view_sizes(case))
        return {"bytes": 17 * rays, "flops": 20 * depth * rays}
    rays = case["width"] * case["height"]
    if kind == "frame":
        return {"bytes": 4 * rays + 4 * (rays // 64), "flops": 20 * depth * rays}
    if kind == "shadow":
        return {"bytes": 18 * rays, "flops": 40 * depth * rays}
    return {"bytes": 17 * rays, "flops": 20 * depth * rays}


# ---- 64-bit values ------------------------------------------------------------


def _first_hits(occ, res, o, d):
    """Entry distance of each ray into the first occupied voxel of the dense
    res^3 volume over [1,2]^3 (0 where none), stepped in float64."""
    d = torch.where(d.abs() < 1e-4, torch.full_like(d, 1e-4), d)
    near = ((torch.where(d > 0, 1.0, 2.0) - o) / d).amax(1).clamp_min(0.0)
    far = ((torch.where(d > 0, 2.0, 1.0) - o) / d).amin(1)
    t = torch.zeros(len(o), dtype=torch.float64, device=o.device)
    live = (near < far).nonzero()[:, 0]
    o, d, now = o[live], d[live], near[live]
    step = torch.sign(d).long()
    cell = ((o + d * now[:, None] - 1.0) * res).floor().long().clamp(0, res - 1)
    edge = (step > 0).double()
    while len(live):
        hit = occ[cell[:, 2], cell[:, 1], cell[:, 0]]
        t[live[hit]] = now[hit]
        nxt = ((cell.double() + edge) / res + 1.0 - o) / d
        now, axis = nxt.min(1)
        cell = cell.scatter_add(1, axis[:, None], step.gather(1, axis[:, None]))
        on = ~hit & (cell >= 0).all(1) & (cell < res).all(1)
        live, o, d, now, cell, step, edge = live[on], o[on], d[on], now[on], cell[on], step[on], edge[on]
    return t


def _primary_rays(m, pos, w, h):
    """The image's rays in float64; a direction is scaled by the image plane's
    inverse square root (one Newton step from the bit-level first guess)."""
    m = torch.from_numpy(m.astype(np.float64)).cuda()
    y, x = torch.meshgrid(torch.arange(h, device="cuda").double(), torch.arange(w, device="cuda").double(),
                          indexing="ij")
    dx, dy = (x * 2.0 / w - 1.0).reshape(-1, 1), (h / w - y * 2.0 / w).reshape(-1, 1)
    v = dx * m[:3, 0] + dy * m[:3, 1] + m[:3, 2] / math.tan(math.pi / 6.0)
    q = (v * v).sum(1)
    guess = (0x5F3759DF - (q.float().view(torch.int32) >> 1)).view(torch.float32).double()
    d = v * (guess * (1.5 - 0.5 * q * guess * guess))[:, None]
    return torch.from_numpy(pos.astype(np.float64)).cuda().expand_as(d), d


def exact(case, seed):
    """Entry distances of the dense-volume scenes; the other outputs are whole
    numbers (hit codes, leaf words and indices, octree words, file bytes), and
    the other scenes have no dense volume to step through in seconds."""
    if case["kind"] not in ("rays", "primary") or case["scene"] != "grid" or case.get("lod"):
        return None
    res = case["res"]
    if case["kind"] == "rays":
        o, d, _ = _query_rays(case, seed)
        o, d = o.double(), d.double()
    else:
        rng = np.random.default_rng(seed + 3)
        o, d = _primary_rays(*_camera(rng, case["scene"]), case["width"], case["height"])
    occ = _volume(seed, res, res, res, res) != 0
    return {"hit": None, "normal": None, "t": _first_hits(occ, res, o, d), "leaf": None}
