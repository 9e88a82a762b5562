"""Unit boxes: a frame draws only the units of a mesh that its view may see.

crx_mesh_create computes an object-space box per stage-1 unit (8 rows of 128
triangles) of meshes of 2^20 triangles and more; k_cull_units lists the units
a view may see and marks those wholly inside it, and k_stage1_pairs walks the
list, cut into parts of 1 to 8 rows.  A dropped unit holds no triangle that
its own tests would keep, so every frame must equal the walk over all
triangles (stage1_layout = 0, which uses no boxes) and the oracle bit for bit
(tolerance: none): for views that see everything, a corner, nothing, from
inside the terrain and across the near plane; for rows, shuffled,
non-indexed and IX_PU16 meshes, several instances, mirrors and non-finite
vertices; through a recorded frame; and after the geometry was handed out and
rewritten.
"""
import ctypes as C

import numpy as np
import pytest

import crx
import oracle as orc
import workloads as wl
from crxtest import describe_mismatch

pytestmark = pytest.mark.gpu

N = 801     # 1.28 M triangles, rows of 1600
W, H = 500, 300


@pytest.fixture(scope="module")
def ctx():
    c = crx.Context(0)
    yield c
    c.close()


@pytest.fixture(scope="module")
def terrain():
    return wl.heightfield_mesh(N, amplitude=20.0, scale=100.0)


def _views():
    c = 0.5 * (N - 1)
    up = (0.0, 1.0, 0.0)
    return {
        "whole": crx.look_at((c, 1.1 * N, c - 0.4 * N), (c, 0.0, c), (0.0, 0.0, 1.0)),
        "edge": crx.look_at((c, 60.0, -40.0), (c, 30.0, 0.0), up),
        "corner": crx.look_at((-30.0, 40.0, -30.0), (10.0, 0.0, 12.0), up),
        "away": crx.look_at((c, 60.0, -40.0), (c, 60.0, -400.0), up),
        "inside": crx.look_at((c, 0.5, c), (c + 10.0, 0.0, c + 30.0), up),
        "below": crx.look_at((c, -50.0, c), (c + 1.0, 40.0, c), (0.0, 0.0, 1.0)),
    }


def _frame(ctx, scene, view, boxes, w=W, h=H):
    t = crx.default_tuning()
    if not boxes:
        t.stage1_layout = 0
    ctx.tuning = t
    try:
        fb, cb = ctx.alloc(8 * w * h), ctx.alloc(8 * w * h)
        st = scene.render(crx.make_view(view, wl.projection(w, h), w, h), fb, cb, crx.render_settings())
        out = fb.download(np.uint64, w * h), cb.download(np.uint64, w * h)
        fb.free()
        cb.free()
        # (a view away from the mesh's own box draws no node at all)
        assert st.stage1_kernel == (2 if boxes and st.num_triangles else 0)
        return out
    finally:
        ctx.tuning = crx.default_tuning()


def _same(a, b, w=W):
    assert np.array_equal(a[0], b[0]), describe_mismatch(a[0], b[0], w)
    assert np.array_equal(a[1], b[1]), describe_mismatch(a[1], b[1], w)


@pytest.mark.parametrize("form", ["rows", "shuffled", "plain", "packed"])
def test_listed_units_equal_the_whole_walk(ctx, terrain, form):
    pos, idx, col = terrain
    if form == "shuffled":
        idx = idx[np.random.default_rng(5).permutation(len(idx))]
    mesh = (crx.Mesh(ctx, pos[idx.reshape(-1)], None, col[idx.reshape(-1)]) if form == "plain"
            else crx.Mesh(ctx, pos, idx, col, compressed=form == "packed"))
    scene = crx.Scene(ctx)
    scene.add(mesh)
    for name, view in _views().items():
        got, want = _frame(ctx, scene, view, True), _frame(ctx, scene, view, False)
        _same(got, want)
        assert (got[0] != crx.CLEAR_PIXEL).any() == (name not in ("away", "below"))
    scene.close()
    mesh.close()


def test_against_the_oracle(ctx, terrain):
    pos, idx, col = terrain
    mesh = crx.Mesh(ctx, pos, idx, col)
    scene = crx.Scene(ctx)
    scene.add(mesh)
    m = crx.CMesh()
    m.numTriangles, m.numVertices, m.isLoaded = len(idx), len(pos), 1
    m.positions, m.indices, m.colors = pos.ctypes.data, idx.ctypes.data, col.ctypes.data
    m.instances.count = 1
    m.world = crx.identity()
    proj = wl.projection(W, H)
    for name in ("edge", "inside"):
        view = _views()[name]
        xf = [crx.mat4_mul(view, crx.identity())]
        fb, _ = orc.draw(crx, [m], [m], xf, W, H, view, proj, False)
        got = _frame(ctx, scene, view, True)
        assert np.array_equal(got[0], fb), describe_mismatch(got[0], fb, W)
    scene.close()
    mesh.close()


def test_instances_mirrors_and_non_finite(ctx, terrain):
    pos, idx, col = terrain
    bad = pos.copy()
    rng = np.random.default_rng(8)
    for k in rng.integers(0, len(bad), 40):
        bad[k, int(rng.integers(3))] = rng.choice([np.nan, np.inf, -np.inf])
    mirror = np.diag([-1.0, 1.0, 1.0, 1.0]).astype(np.float32)
    mirror[:3, 3] = (N - 1.0, 5.0, 30.0)
    small = crx.Mesh(ctx, *wl.sphere_mesh(40, 60, radius=30.0))      # a mesh without boxes in the same draw
    meshes = [crx.Mesh(ctx, pos, idx, col), crx.Mesh(ctx, bad, idx, col), small]
    scene = crx.Scene(ctx)
    scene.add(meshes[0])
    scene.add(meshes[0], crx.Mat4.from_numpy(mirror))
    scene.add(meshes[1], crx.Mat4.from_numpy(mirror))
    scene.add(small)
    for view in _views().values():
        a, b = _frame(ctx, scene, view, True), _frame(ctx, scene, view, False)
        _same(a, b)
    scene.close()
    for m in meshes:
        m.close()


def test_recorded_frame_and_handed_out_geometry(ctx, terrain):
    pos, idx, col = terrain
    mesh = crx.Mesh(ctx, pos, idx, col)
    scene = crx.Scene(ctx)
    scene.add(mesh)
    views = list(_views().values())
    fb, cb = ctx.alloc(8 * W * H), ctx.alloc(8 * W * H)
    v = [crx.make_view(x, wl.projection(W, H), W, H) for x in views]
    frame = crx.Frame(scene, [v[0]], [fb], [cb])

    def replay(k):
        frame.set_views([v[k]])
        frame.launch()
        frame.wait()
        return fb.download(np.uint64, W * H), cb.download(np.uint64, W * H)

    for k in range(len(views)):
        _same(replay(k), _frame(ctx, scene, views[k], False))
    # the geometry's addresses go out and the vertices move: the boxes no longer count
    p, _, _ = mesh.buffers()
    moved = np.ascontiguousarray(pos + np.array([0.0, 25.0, -60.0], dtype=np.float32))
    crx._check(crx.lib().crx_memcpy_htod(ctx.handle, C.c_void_p(p), C.c_void_p(moved.ctypes.data), moved.nbytes, None))
    frame.launch()          # the last view again
    frame.wait()
    last = _frame(ctx, scene, views[-1], False)
    _same((fb.download(np.uint64, W * H), cb.download(np.uint64, W * H)), last)
    for k in range(len(views)):
        want = _frame(ctx, scene, views[k], False)
        _same(replay(k), want)
    frame.close()
    scene.close()
    mesh.close()
    fb.free()
    cb.free()
