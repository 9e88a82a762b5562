"""Stage 1 of several views from one unit list (k_cull_units, k_stage1_pairs).

A draw of several views of meshes that hold unit boxes lists each unit once
for every view that may see it and draws it there in squares of 8 rows of 8
pairs (IX_PU16 meshes row by row).  Only who draws a triangle changes: every
view's buffers equal the oracle's bit for bit (tolerance: none) on grids whose
rows and row count are not whole squares, without row structure, without
indices, compressed, mirrored and repeated, at one list part per unit and at
several, for views of mixed sizes that see all, some or nothing of the mesh and
from close up, and in a recorded frame.
"""
import numpy as np
import pytest

import crx
import oracle as orc
import workloads as wl
from crxtest import CompressedMesh, SceneSpec, describe_mismatch, oracle_render

pytestmark = pytest.mark.gpu

N = 741      # 2 * 740 * 740 = 1,095,200 triangles, past the size from which units have boxes


@pytest.fixture(scope="module")
def ctx():
    c = crx.Context(0)
    yield c
    c.close()


def _grid():
    return wl.heightfield_mesh(N, amplitude=25.0, scale=180.0)


def _views(count):
    c = 0.5 * N
    poses = [((c, 1.1 * N, c - 1.0), (c, 0.0, c)), ((40.0, 60.0, -80.0), (c, 0.0, c)),
             ((c, 30.0, c), (c + 40.0, 0.0, c + 30.0)), ((-50.0, 40.0, -50.0), (-400.0, 40.0, -300.0)),
             ((N - 5.0, 27.0, N - 5.0), (0.0, 0.0, 0.0))]
    sizes = [(320, 200), (101, 77), (640, 360), (257, 33), (480, 480)]
    out = []
    for k in range(count):
        eye, at = poses[k % 5]
        W, H = sizes[(k // 2) % 5]
        out.append((W, H, crx.look_at(eye, (at[0] + 3.0 * (k // 5), at[1], at[2]), (0.0, 1.0, 0.0)), wl.projection(W, H)))
    return out


def _draw(ctx, nodes, views, frame=False):
    scene = crx.Scene(ctx)
    for mesh, world in nodes:
        scene.add(mesh, world)
    vs = [crx.make_view(v, p, W, H) for W, H, v, p in views]
    fbs, cbs = ([ctx.alloc(8 * W * H) for W, H, _, _ in views] for _ in range(2))
    settings = crx.render_settings()
    try:
        if frame:
            f = crx.Frame(scene, vs, fbs, cbs, settings)
            for _ in range(3):
                f.launch()
                f.wait()
            f.close()
            st = None
        else:
            st = scene.render_views(vs, fbs, cbs, settings)
        return [b.download(np.uint64, W * H) for b, (W, H, _, _) in zip(fbs, views)], st
    finally:
        for b in fbs + cbs:
            b.free()
        scene.close()


def _check(ctx, spec, nodes, views, frame=False):
    got, st = _draw(ctx, nodes, views, frame)
    assert st is None or st.stage1_kernel == 2
    for (W, H, view, proj), fb in zip(views, got):
        want, _, _ = oracle_render(spec, W, H, view, proj)
        assert np.array_equal(fb, want), describe_mismatch(fb, want, W)
    assert any((fb != crx.CLEAR_PIXEL).any() for fb in got)


@pytest.mark.parametrize("kind", ["rows", "shuffled", "flat", "compressed"])
@pytest.mark.parametrize("count", [2, 13])
def test_formats(ctx, kind, count):
    pos, idx, _ = _grid()
    if kind == "shuffled":
        idx = idx[np.random.default_rng(4).permutation(len(idx))]
    host = (CompressedMesh(pos, idx) if kind == "compressed" else
            orc.HostMesh(crx, pos[idx.reshape(-1)], None, None) if kind == "flat" else orc.HostMesh(crx, pos, idx, None))
    mesh = (crx.Mesh(ctx, pos, idx, compressed=True) if kind == "compressed" else
            crx.Mesh(ctx, pos[idx.reshape(-1)], None) if kind == "flat" else crx.Mesh(ctx, pos, idx))
    try:
        _check(ctx, SceneSpec().add(host, [crx.identity()]), [(mesh, None)], _views(count))
    finally:
        mesh.close()


@pytest.mark.parametrize("frame", [False, True])
def test_repeated_mirrored_and_small_meshes(ctx, frame):
    """Three instances (one mirrored) of the grid and a mesh without boxes, each seen by some of the views."""
    pos, idx, _ = _grid()
    sp, si, _ = wl.sphere_mesh(40, 60, radius=30.0)
    worlds = []
    for x, z, mirror in ((0.0, 0.0, 1.0), (900.0, 100.0, 1.0), (-300.0, 400.0, -1.0)):
        w = np.diag([mirror, 1.0, 1.0, 1.0]).astype(np.float32)
        w[:3, 3] = (x, 0.0, z)
        worlds.append(crx.Mat4.from_numpy(w))
    ball = np.eye(4, dtype=np.float32)
    ball[:3, 3] = (0.5 * N, 60.0, 0.5 * N)
    ball = crx.Mat4.from_numpy(ball)
    spec = SceneSpec().add(orc.HostMesh(crx, pos, idx, None), worlds).add(orc.HostMesh(crx, sp, si, None), [ball])
    grid, sphere = crx.Mesh(ctx, pos, idx), crx.Mesh(ctx, sp, si)
    try:
        # the spec lists the larger mesh first, as the scene's sort does; every node may be in view
        settings_nodes = [(grid, w) for w in worlds] + [(sphere, ball)]
        far = [((400.0, 1500.0, 300.0), (300.0, 0.0, 400.0)), ((-900.0, 700.0, -800.0), (300.0, 0.0, 300.0)),
               ((300.0, 1800.0, -600.0), (300.0, 0.0, 300.0))]
        views = [(W, H, crx.look_at(e, a, (0.0, 1.0, 0.1)), wl.projection(W, H))
                 for (e, a), (W, H) in zip(far, ((333, 222), (640, 360), (160, 200)))]
        _check(ctx, spec, settings_nodes, views, frame)
    finally:
        grid.close()
        sphere.close()
