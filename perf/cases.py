"""Workloads of the visibility-buffer rasterizer, as a user's program calls it.

Every case is one frame (or one batch of views, or one burst of requests)
through a public entry point: the scene API, the hipGraph frame, the raw
drawTrianglesVisbuffer boundary, the batched views and the out-of-core server.
Outputs are the whole visibility and colour buffers; they are packed integers
(28-bit depth | 36-bit triangle id, and depth | RGBA8).

    listed()             the fixed cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  scene, meshes and buffers on the GPU
    run(state)           one pass; returns the buffers it filled
    work(case)           bytes and operations the frame cannot do without
"""
import math
import os
import sys

import numpy as np
import torch  # before the binding, so that both use one HIP runtime

sys.path.insert(0, os.path.join(os.getcwd(), "curast-ooc_amd"))

import crx  # noqa: E402
import workloads as wl  # noqa: E402

ATTRIBUTES = {"texture": crx.DISPLAY_TEXTURE, "normal": crx.DISPLAY_NORMAL, "uv": crx.DISPLAY_UV,
              "colors": crx.DISPLAY_VERTEX_COLORS, "triangle_id": crx.DISPLAY_TRIANGLE_ID}


def listed():
    return [
        # A preview thumbnail: the smallest frame, bound by launches and latency.
        {"name": "thumbnail_1k", "kind": "sphere", "rings": 16, "segments": 32, "width": 256, "height": 256,
         "attribute": "colors"},
        # One scanned object filling a 1080p window (the repository's small configuration).
        {"name": "sphere_1m_1080p", "kind": "sphere", "rings": 512, "segments": 1024, "width": 1920, "height": 1080,
         "attribute": "colors"},
        # The same frame recorded once and replayed with a new camera each time: an interactive viewer's loop.
        {"name": "graph_sphere_130k_720p", "kind": "graph", "rings": 256, "segments": 256, "width": 1280,
         "height": 720, "attribute": "normal"},
        # A fly-over of a very large terrain held as one mesh: most of it lies outside the view (the headline benchmark).
        {"name": "terrain_400m_1080p", "kind": "terrain", "n": 14142, "camera": "edge", "width": 1920, "height": 1080,
         "attribute": "colors", "compressed": False},
        # An overview of a whole terrain: every triangle is inside the view, most are smaller than a pixel.
        {"name": "terrain_25m_overview", "kind": "terrain", "n": 3537, "camera": "overview", "width": 1280,
         "height": 720, "attribute": "triangle_id", "compressed": False},
        # The memory-saving IX_PU16 format, flown over at an odd size.
        {"name": "terrain_ixpu16_32m", "kind": "terrain", "n": 4001, "camera": "edge", "width": 1917, "height": 1077,
         "attribute": "colors", "compressed": True},
        # Standing on the ground at 4K with textures: medium and huge triangles (stages 2 and 3) and the
        # textured resolve, the reference's default display.
        {"name": "closeup_4k_textured", "kind": "terrain", "n": 1025, "camera": "closeup", "width": 3840,
         "height": 2160, "attribute": "texture", "compressed": False},
        # One dense mesh drawn thousands of times (the repository's instancing configuration).
        {"name": "instances_3000x1m", "kind": "instances", "count": 3000, "rings": 512, "segments": 1024,
         "extent": 200.0, "width": 1920, "height": 1080, "attribute": "colors"},
        # A scene graph of several hundred nodes over meshes of very different sizes, some mirrored.
        {"name": "nodes_600_mixed", "kind": "nodes", "meshes": 24, "nodes": 600, "width": 1365, "height": 769,
         "attribute": "normal"},
        # A host that keeps its own CMesh arrays and calls clear, draw and resolve itself.
        {"name": "raw_draw_40_meshes", "kind": "raw", "meshes": 40, "n": 257, "width": 1600, "height": 900,
         "attribute": "uv"},
        # Many remote views of one terrain in one batch, mixed resolutions, a quarter of them close-ups.
        {"name": "views_64_mixed", "kind": "views", "n": 7072, "views": 64, "attribute": "colors"},
        # A burst of requests to the out-of-core server over 1M-triangle nodes.
        {"name": "serve_burst_32", "kind": "serve", "tiles": 5, "tile": 703, "requests": 32, "attribute": "colors"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sphere", "graph", "terrain", "terrain", "terrain", "instances", "nodes", "raw", "views",
                       "serve"])
    size = {"width": _log(rng, 200, 3840), "height": _log(rng, 150, 2160)}
    attr = rng.choice(["colors", "normal", "triangle_id"])
    if kind in ("sphere", "graph"):
        return {"kind": kind, "rings": _log(rng, 12, 600), "segments": _log(rng, 24, 1200), **size,
                "attribute": attr}
    if kind == "terrain":
        camera = rng.choice(["edge", "edge", "overview", "closeup"])
        compressed = rng.random() < 0.3
        n = _log(rng, 300, 5000 if compressed else 10000)
        if camera == "closeup":
            n = min(n, 3000)
            attr = rng.choice(["texture", "colors"])
        return {"kind": kind, "n": n, "camera": camera, **size, "attribute": attr, "compressed": compressed}
    if kind == "instances":
        return {"kind": kind, "count": _log(rng, 30, 3000), "rings": _log(rng, 40, 512),
                "segments": _log(rng, 80, 1024), "extent": 200.0, **size, "attribute": attr}
    if kind == "nodes":
        return {"kind": kind, "meshes": _log(rng, 4, 40), "nodes": _log(rng, 50, 1500), **size, "attribute": attr}
    if kind == "raw":
        return {"kind": kind, "meshes": _log(rng, 4, 120), "n": _log(rng, 40, 500), **size, "attribute": "uv"}
    if kind == "views":
        return {"kind": kind, "n": _log(rng, 700, 6000), "views": _log(rng, 2, 64), "attribute": "colors"}
    return {"kind": kind, "tiles": rng.randint(3, 5), "tile": _log(rng, 100, 703), "requests": _log(rng, 8, 48),
            "attribute": "colors"}


# ---------------------------------------------------------------------------
# Cameras and scenes
# ---------------------------------------------------------------------------


def _view(camera, n, width, height, ground=None):
    if camera == "edge":
        view, proj = wl.heightfield_view(n, width, height)
    elif camera == "overview":
        c = 0.5 * (n - 1)
        # far enough back that the whole square lies inside both fields of view
        reach = 1.05 * n * max(1.0, height / width)
        view = crx.look_at((c, reach, c - 0.45 * reach), (c, 0.0, c), (0.0, 0.0, 1.0))
        proj = wl.projection(width, height)
    else:  # standing on the ground, looking down at the cells in front
        c = int(0.4 * n)
        eye = (c + 0.5, ground + 2.0, c + 0.5)
        view = crx.look_at(eye, (eye[0] + 0.3, eye[1] - 0.55, eye[2] + 1.0), (0.0, 1.0, 0.0))
        proj = wl.projection(width, height)
    return view, proj


class _Ptr:
    """A device buffer of the caller's own (a tensor), as the binding takes it."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = tensor.data_ptr()


def _buffer(pixels):
    return _Ptr(torch.zeros(pixels, dtype=torch.int64, device="cuda"))


class State:
    """What the user's program keeps: context, meshes, scene and its buffers."""

    def __init__(self, case):
        self.case = case
        self.ctx = crx.Context(0)
        self.keep = []      # closed in reverse order, before the context
        self.meshes = []

    def mesh(self, *args, **kw):
        m = crx.Mesh(self.ctx, *args, **kw)
        self.meshes.append(m)
        return m

    def close(self):
        if self.ctx is None:
            return
        torch.cuda.synchronize()
        for x in reversed(self.keep):
            x()
        for m in self.meshes:
            m.close()
        self.ctx.close()
        self.ctx = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


def _scene(st, nodes):
    scene = crx.Scene(st.ctx)
    st.keep.append(scene.close)
    for mesh, world in nodes:
        scene.add(mesh, world)
    return scene


def _frame_buffers(st, width, height):
    st.fb, st.cb = _buffer(width * height), _buffer(width * height)


def _settings(case):
    return crx.render_settings(attribute=ATTRIBUTES[case["attribute"]])


def _terrain(n, seed, shape):
    """Height noise with a wavelength that scales with small terrains, so that each has hills."""
    scale = min(2048.0, n / 4.0) if shape != "closeup" else 64.0
    return wl.heightfield_mesh(n, amplitude=min(120.0, scale / 8.0), scale=scale, seed=wl.SEED_HEIGHTFIELD + seed)


def _prepare_sphere(st, case, seed):
    W, H = case["width"], case["height"]
    pos, idx, col = wl.sphere_mesh(case["rings"], case["segments"], seed=wl.SEED_SPHERE + seed)
    scene = _scene(st, [(st.mesh(pos, idx, col), None)])
    view, proj = wl.sphere_view(W, H)
    _frame_buffers(st, W, H)
    st.view = crx.make_view(view, proj, W, H)
    st.scene, st.settings = scene, _settings(case)


def _prepare_graph(st, case, seed):
    _prepare_sphere(st, case, seed)
    st.frame = crx.Frame(st.scene, [st.view], [st.fb], [st.cb], st.settings)
    st.keep.append(st.frame.close)


def _prepare_terrain(st, case, seed):
    n, W, H = case["n"], case["width"], case["height"]
    pos, idx, col = _terrain(n, seed, case["camera"])
    k = int(0.4 * n)
    view, proj = _view(case["camera"], n, W, H, float(pos[k * n + k, 1]))
    mesh = st.mesh(pos, idx, col, compressed=case["compressed"])
    scene = _scene(st, [(mesh, None)])
    if case["attribute"] == "texture":
        size = 2048
        rng = np.random.default_rng(seed)
        uv = (pos[:, [0, 2]] / 16.0).astype(np.float32)
        mesh.set_attributes(uvs=uv)
        chain = torch.zeros(crx.texture_chain_texels(size, size), dtype=torch.int32, device="cuda")
        level0 = rng.integers(0, 1 << 24, size * size, dtype=np.int32)
        chain[:size * size] = torch.from_numpy(level0).cuda()
        st.ctx.compute_mipmap(chain.data_ptr(), size, size)
        tex = crx.Texture()
        tex.width, tex.height, tex.data = size, size, chain.data_ptr()
        scene.set_texture(0, tex)
        st.chain = chain
    _frame_buffers(st, W, H)
    st.view = crx.make_view(view, proj, W, H)
    st.scene, st.settings = scene, _settings(case)


def _prepare_instances(st, case, seed):
    W, H = case["width"], case["height"]
    pos, idx, col = wl.sphere_mesh(case["rings"], case["segments"], seed=wl.SEED_SPHERE + seed)
    mesh = st.mesh(pos, idx, col)
    worlds = wl.instance_transforms(case["count"], extent=case["extent"], seed=wl.SEED_INSTANCES + seed)
    scene = _scene(st, [(mesh, w) for w in worlds])
    view, proj = wl.instances_view(case["extent"], W, H)
    _frame_buffers(st, W, H)
    st.view = crx.make_view(view, proj, W, H)
    st.scene, st.settings = scene, _settings(case)


def _mesh_sizes(count):
    """Sphere sizes of a scene's meshes: from 200 to about 200,000 triangles."""
    out = []
    for k in range(count):
        rings = int(round(10 * (32.0 ** (k / max(1, count - 1)))))
        out.append((rings, rings))
    return out


def _prepare_nodes(st, case, seed):
    W, H = case["width"], case["height"]
    meshes = [st.mesh(*wl.sphere_mesh(r, s, seed=wl.SEED_SPHERE + 100 * seed + k))
              for k, (r, s) in enumerate(_mesh_sizes(case["meshes"]))]
    worlds = list(wl.instance_transforms(case["nodes"], extent=30.0, seed=wl.SEED_INSTANCES + seed))
    rng = np.random.default_rng(seed)
    nodes = []
    for w in worlds:
        if rng.random() < 0.2:      # a mirrored copy
            for e in range(4):
                w.m[e] = -w.m[e]
        nodes.append((meshes[int(rng.integers(len(meshes)))], w))
    scene = _scene(st, nodes)
    view = crx.look_at((15.0, 18.0, -12.0), (15.0, 12.0, 15.0), (0.0, 1.0, 0.0))
    _frame_buffers(st, W, H)
    st.view = crx.make_view(view, wl.projection(W, H), W, H)
    st.scene, st.settings = scene, _settings(case)


def _prepare_raw(st, case, seed):
    n, W, H, count = case["n"], case["width"], case["height"], case["meshes"]
    view = crx.look_at((-4.0, 30.0, -20.0), (30.0, 0.0, 40.0), (0.0, 1.0, 0.0))
    proj = wl.projection(W, H)
    instances, transforms, prefix, total = [], [], [], 0
    side = int(math.ceil(math.sqrt(count)))
    for k in range(count):
        pos, idx, _ = wl.heightfield_mesh(n, spacing=10.0 / n, amplitude=0.6, scale=2.0,
                                          seed=wl.SEED_HEIGHTFIELD + 1000 * seed + k)
        uv = (pos[:, [0, 2]] / 10.0).astype(np.float32)
        bufs = [torch.from_numpy(pos).cuda(), torch.from_numpy(idx.view(np.int32)).cuda(), torch.from_numpy(uv).cuda()]
        st.keep.append(lambda b=bufs: b.clear())
        world = np.eye(4, dtype=np.float32)
        world[:3, 3] = (11.0 * (k % side), 0.0, 11.0 * (k // side))
        m = crx.CMesh()
        m.numTriangles, m.numVertices = len(idx), len(pos)
        m.positions, m.indices, m.uvs = (b.data_ptr() for b in bufs)
        m.cummulativeTriangleCount = total
        m.instances.offset, m.instances.count = k, 1
        m.world = crx.Mat4.from_numpy(world)
        m.id, m.isLoaded = k, 1
        instances.append(m)
        transforms.append(crx.mat4_mul(view, m.world))
        prefix.append(total)
        total += len(idx)
    st.instances = (crx.CMesh * count)(*instances)
    st.transforms = (crx.Mat4 * count)(*transforms)
    st.prefix = np.array(prefix, dtype=np.uint64)
    _frame_buffers(st, W, H)
    st.target = crx.make_target(st.fb.ptr, st.cb.ptr, W, H, view, proj)


def _prepare_views(st, case, seed):
    n = case["n"]
    pos, idx, col = _terrain(n, seed, "views")
    scene = _scene(st, [(st.mesh(pos, idx, col), None)])
    # the resolutions are the case's own, the cameras the seed's
    sizes = [wl.MULTIVIEW_SIZES[k % len(wl.MULTIVIEW_SIZES)] for k in range(case["views"])]
    poses = wl.multiview_views(n, pos, count=case["views"], sizes=((1920, 1080),), seed=wl.SEED_VIEWS + seed)
    total = sum(w * h for w, h in sizes)
    st.fb, st.cb = _buffer(total), _buffer(total)
    st.views, st.fbs, st.cbs, at = [], [], [], 0
    for (view, _, _, _, _), (w, h) in zip(poses, sizes):
        st.views.append(crx.make_view(view, wl.projection(w, h), w, h))
        st.fbs.append(_Ptr(st.fb.tensor[at:at + w * h]))
        st.cbs.append(_Ptr(st.cb.tensor[at:at + w * h]))
        at += w * h
    st.scene, st.settings = scene, _settings(case)


SERVE_SIZES = ((256, 256), (512, 512), (1280, 720), (1920, 1080))


def _prepare_serve(st, case, seed):
    tile = case["tile"]
    n = case["tiles"] * tile + 1
    nodes, buffers = wl.tiled_heightfield(st.ctx, n, tile, amplitude=60.0, scale=512.0, chunk_bytes=1 << 26,
                                          seed=wl.SEED_HEIGHTFIELD + seed)
    for b in buffers:
        st.keep.append(b.free)
    up = lambda x: (x + 255) // 256 * 256  # noqa: E731
    slot = max(up(12 * d["nv"]) + up(12 * d["nt"]) + up(4 * d["nv"]) for d in nodes)
    # the device holds four fifths of the nodes
    cfg = crx.server_config(node_cache_bytes=slot * max(4, len(nodes) * 4 // 5), frame_bytes=2 << 30,
                            max_batch_views=64, lanes=2, resolve=1)
    srv = crx.Server(st.ctx, cfg)
    st.keep.append(srv.close)
    for d in nodes:
        srv.add_node(d["pos"], d["nv"], d["idx"], d["nt"], d["col"], d["aabb"])
    srv.start()
    ground = wl.ground_lookup(nodes, tile)
    stream = wl.serving_requests(n, ground, duration=1.0 + case["requests"] / 100.0, rate=200.0, sessions=4,
                                 seed=wl.SEED_SERVING + seed)[:case["requests"]]
    st.views, total = [], 0
    for k, (_, view, _, _, _, _) in enumerate(stream):
        w, h = SERVE_SIZES[k % len(SERVE_SIZES)]
        st.views.append(crx.make_view(view, wl.projection(w, h), w, h))
        total += w * h
    st.server = srv
    st.fb, st.cb = _buffer(total), _buffer(total)


PREPARE = {"sphere": _prepare_sphere, "graph": _prepare_graph, "terrain": _prepare_terrain,
           "instances": _prepare_instances, "nodes": _prepare_nodes, "raw": _prepare_raw, "views": _prepare_views,
           "serve": _prepare_serve}


def prepare(case, seed):
    st = State(case)
    PREPARE[case["kind"]](st, case, seed % 100003)
    return st


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------


class _At:
    """A device address handed to the binding's copy."""

    def __init__(self, ptr):
        self.ptr = ptr


def run(st):
    case = st.case
    kind = case["kind"]
    if kind == "graph":
        st.frame.set_views([st.view])
        st.frame.launch()
        st.frame.wait()
    elif kind == "raw":
        pixels = case["width"] * case["height"]
        st.ctx.clear_framebuffer(st.fb.ptr, pixels)
        st.ctx.clear_framebuffer(st.cb.ptr, pixels)
        st.ctx.draw_triangles_visbuffer(st.instances, st.instances, st.transforms, st.target, False)
        st.ctx.resolve_visbuffer(st.instances, st.prefix, st.target, ATTRIBUTES[case["attribute"]])
    elif kind == "views":
        st.scene.render_views(st.views, st.fbs, st.cbs, st.settings)
    elif kind == "serve":
        tickets = [st.server.submit(v) for v in st.views]
        at = 0
        for ticket, v in zip(tickets, st.views):
            r = st.server.wait(ticket)
            if r.status != 0:
                raise RuntimeError("request failed")
            px = v.width * v.height
            # the user keeps each frame on the device (an encoder reads it there)
            st.ctx.copy(_At(st.fb.ptr + 8 * at), _At(r.framebuffer), 8 * px)
            st.ctx.copy(_At(st.cb.ptr + 8 * at), _At(r.colorbuffer), 8 * px)
            at += px
        st.ctx.synchronize()   # the results' memory goes back to the server
        for ticket in tickets:
            st.server.release(ticket)
    else:
        st.scene.render(st.view, st.fb, st.cb, st.settings)
    return {"visibility": st.fb.tensor, "color": st.cb.tensor}


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------


def _seen(n, views):
    """Share of a flat n x n terrain that any of the (view, proj) cameras sees, from 256 x 256 sample points."""
    g = np.linspace(0.0, n - 1.0, 256)
    x, z = np.meshgrid(g, g)
    p = np.stack([x.ravel(), np.zeros(x.size), z.ravel(), np.ones(x.size)])
    seen = np.zeros(x.size, dtype=bool)
    for view, proj in views:
        v = np.array(view.m, dtype=np.float64).reshape(4, 4).T @ p
        pm = np.array(proj.m, dtype=np.float64).reshape(4, 4)
        d = -v[2]
        with np.errstate(all="ignore"):
            seen |= (d > 0) & (np.abs(pm[0, 0] * v[0]) <= d) & (np.abs(pm[1, 1] * v[1]) <= d)
    return max(float(seen.mean()), 1.0 / p.shape[1])


def work(case):
    """Bytes: indices and positions of the triangles inside the view read once, the visibility and the colour
    buffer written once (and the visibility buffer read once by the resolve).  Operations: the transform and
    edge setup (about 120) of each triangle inside the view, taken once per instance at most once per pixel a
    dense instance covers, and about 200 per shaded pixel."""
    kind = case["kind"]
    shade = 400.0 if case["attribute"] == "texture" else 200.0
    if kind in ("terrain", "views"):
        n = case["n"]
        tris, verts = 2.0 * (n - 1) ** 2, float(n) * n
        if kind == "terrain":
            px = float(case["width"] * case["height"])
            share = _seen(n, [_view(case["camera"], n, case["width"], case["height"], 0.0)])
        else:
            sizes = [wl.MULTIVIEW_SIZES[k % len(wl.MULTIVIEW_SIZES)] for k in range(case["views"])]
            px = float(sum(w * h for w, h in sizes))
            flat = np.zeros((n * n, 3), dtype=np.float32)
            poses = wl.multiview_views(n, flat, count=case["views"], sizes=((1920, 1080),))
            share = _seen(n, [(p[0], wl.projection(w, h)) for p, (w, h) in zip(poses, sizes)])
        bits = math.ceil(math.log2(verts)) if case.get("compressed") else 32
        geo = share * (tris * 3 * bits / 8 + verts * (6 if case.get("compressed") else 12))
        return {"bytes": geo + 24.0 * px, "flops": 120.0 * share * tris + shade * px}
    if kind in ("sphere", "graph"):
        px = float(case["width"] * case["height"])
        tris, verts = 2.0 * case["rings"] * case["segments"], (case["rings"] + 1.0) * case["segments"]
        return {"bytes": 12 * tris + 12 * verts + 24 * px, "flops": 120 * tris + shade * 0.35 * px}
    if kind == "instances":
        px = float(case["width"] * case["height"])
        tris, verts = 2.0 * case["rings"] * case["segments"], (case["rings"] + 1.0) * case["segments"]
        return {"bytes": 12 * tris + 12 * verts + 64.0 * case["count"] + 24 * px,
                "flops": 120.0 * min(tris * case["count"], 8.0 * px) + shade * px}
    if kind == "nodes":
        px = float(case["width"] * case["height"])
        tris = sum(2.0 * r * s for r, s in _mesh_sizes(case["meshes"]))
        return {"bytes": 18 * tris + 64.0 * case["nodes"] + 24 * px,
                "flops": 120.0 * tris * case["nodes"] / case["meshes"] + shade * px}
    if kind == "raw":
        px = float(case["width"] * case["height"])
        tris = 2.0 * (case["n"] - 1) ** 2 * case["meshes"]
        return {"bytes": 18 * tris + 32 * px, "flops": 120 * tris + shade * px}
    px = float(sum(w * h for w, h in (SERVE_SIZES[k % len(SERVE_SIZES)] for k in range(case["requests"]))))
    tris = 2.0 * (case["tiles"] * case["tile"]) ** 2
    share = 0.25        # four cameras low over the terrain
    return {"bytes": 18 * share * tris + (24.0 + 32.0) * px, "flops": 120 * share * tris + shade * px}
