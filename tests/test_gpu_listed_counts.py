"""Each triangle of a draw from a unit list is drawn once.

k_stage1_pairs cuts the units that k_cull_units lists into parts of 1 to 8
rows.  A minimum is the same however often it is taken, so the buffers do not
show a row that two parts draw; the stage-2 and stage-3 counts do.  They must
equal the oracle's (tolerance: none) on meshes whose rows are no whole number
of units and whose last rows hold near-plane triangles in view, at every
number of parts, with a mesh of long rows and no boxes in the same draw, for
IX_PU16 meshes in several views, and in a recorded frame whose queues hold
exactly the real entries, before and after its geometry was handed out.
"""
import numpy as np
import pytest

import crx
import oracle as orc
import workloads as wl
from crxtest import CompressedMesh, SceneSpec, describe_mismatch, oracle_render

pytestmark = pytest.mark.gpu

W, H = 400, 300
COLS = 600     # quads per row: 1200 triangles, rows long enough for strips


@pytest.fixture(scope="module")
def ctx():
    c = crx.Context(0)
    yield c
    c.close()


def _grid(rows, cols=COLS, z0=0.0):
    """rows x cols unit quads with a gentle height field, row by row."""
    z, x = np.meshgrid(np.arange(rows + 1, dtype=np.float32), np.arange(cols + 1, dtype=np.float32), indexing="ij")
    y = (0.3 * np.sin(0.21 * x + 0.13 * z)).astype(np.float32)
    pos = np.stack([x - 0.5 * cols, y, z + z0], axis=2).reshape(-1, 3).astype(np.float32)
    a = (np.arange(rows, dtype=np.uint32)[:, None] * np.uint32(cols + 1) + np.arange(cols, dtype=np.uint32)).reshape(-1)
    b, c, d = a + np.uint32(1), a + np.uint32(cols + 1), a + np.uint32(cols + 2)
    return pos, np.stack([a, c, d, a, d, b], axis=1).reshape(-1, 3)


def _edge_view(rows, x=0.0):
    """From just inside the last row, low over it, towards the first."""
    return crx.look_at((x, 1.0, rows + 0.5), (x, 0.2, rows - 6.0), (0.0, 1.0, 0.0))


def _render(ctx, nodes, view, listed, w=W, h=H):
    t = crx.default_tuning()
    if not listed:
        t.stage1_layout = 0
    ctx.tuning = t
    scene = crx.Scene(ctx)
    fb, cb = ctx.alloc(8 * w * h), ctx.alloc(8 * w * h)
    try:
        for mesh, world in nodes:
            scene.add(mesh, world)
        st = scene.render(crx.make_view(view, wl.projection(w, h), w, h), fb, cb, crx.render_settings())
        return fb.download(np.uint64, w * h), st
    finally:
        ctx.tuning = crx.default_tuning()
        scene.close()
        fb.free()
        cb.free()


def _counts(st):
    return st.num_nontrivial, st.num_huge


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("rows", [877, 880, 881])     # 5, 8 and 1 rows in the last unit
def test_counts_of_the_last_rows(ctx, rows, packed):
    pos, idx = _grid(rows)
    host = CompressedMesh(pos, idx) if packed else orc.HostMesh(crx, pos, idx, None)
    mesh = crx.Mesh(ctx, pos, idx, compressed=packed)
    try:
        assert mesh.num_triangles >= 1 << 20 and mesh.row_triangles() == 2 * COLS
        view = _edge_view(rows)
        want, _, st = oracle_render(SceneSpec().add(host, [crx.identity()]), W, H, view, wl.projection(W, H))
        fb, gst = _render(ctx, [(mesh, None)], view, True)
        assert gst.stage1_kernel == 2 and st.num_nontrivial > 50 and st.num_huge > 0
        assert np.array_equal(fb, want), describe_mismatch(fb, want, W)
        assert _counts(gst) == _counts(st)
    finally:
        mesh.close()


@pytest.mark.parametrize("rows", [877, 9005, 18003, 42003])
def test_counts_at_every_number_of_parts(ctx, rows):
    """1.05, 10.8, 21.6 and 50.4 M triangles, made narrow so that the view sees
    almost all of them: 8, 4, 2 and 1 parts per unit on 256 CUs, against the walk
    over all triangles."""
    pos, idx = _grid(rows)
    mesh = crx.Mesh(ctx, pos, idx)
    squash = crx.Mat4.from_numpy(np.diag([0.02, 1.0, 1.0, 1.0]).astype(np.float32))
    try:
        view = _edge_view(rows)
        want, wst = _render(ctx, [(mesh, squash)], view, False)
        fb, gst = _render(ctx, [(mesh, squash)], view, True)
        assert gst.stage1_kernel == 2 and wst.stage1_kernel != 2 and wst.num_nontrivial > 50
        assert np.array_equal(fb, want), describe_mismatch(fb, want, W)
        assert _counts(gst) == _counts(wst)
    finally:
        mesh.close()


def test_counts_with_a_mesh_without_boxes(ctx):
    """A mesh of long rows and too few triangles for boxes: all of its units are
    listed, the empty ones that pad its strips among them."""
    rows, few = 880, 10
    pos, idx = _grid(rows)
    sp, si = _grid(few, z0=float(rows))
    big, small = crx.Mesh(ctx, pos, idx), crx.Mesh(ctx, sp, si)
    try:
        assert small.row_triangles() == 2 * COLS
        spec = (SceneSpec().add(orc.HostMesh(crx, pos, idx, None), [crx.identity()])
                .add(orc.HostMesh(crx, sp, si, None), [crx.identity()]))
        view = _edge_view(rows + few)
        want, _, st = oracle_render(spec, W, H, view, wl.projection(W, H))
        fb, gst = _render(ctx, [(big, None), (small, None)], view, True)
        assert gst.stage1_kernel == 2 and st.num_nontrivial > 50
        assert np.array_equal(fb, want), describe_mismatch(fb, want, W)
        assert _counts(gst) == _counts(st)
    finally:
        big.close()
        small.close()


@pytest.mark.parametrize("packed", [False, True])
def test_counts_of_several_views(ctx, packed):
    rows = 877
    pos, idx = _grid(rows)
    host = CompressedMesh(pos, idx) if packed else orc.HostMesh(crx, pos, idx, None)
    mesh = crx.Mesh(ctx, pos, idx, compressed=packed)
    scene = crx.Scene(ctx)
    scene.add(mesh)
    views = [(W, H, _edge_view(rows, x), wl.projection(W, H)) for x in (-200.0, 3.0, 150.0)]
    fbs, cbs = ([ctx.alloc(8 * W * H) for _ in views] for _ in range(2))
    try:
        gst = scene.render_views([crx.make_view(v, p, w, h) for w, h, v, p in views], fbs, cbs, crx.render_settings())
        assert gst.stage1_kernel == 2
        nt = hg = 0
        for (w, h, v, p), fb in zip(views, fbs):
            want, _, st = oracle_render(SceneSpec().add(host, [crx.identity()]), w, h, v, p)
            got = fb.download(np.uint64, w * h)
            assert np.array_equal(got, want), describe_mismatch(got, want, w)
            nt, hg = nt + st.num_nontrivial, hg + st.num_huge
        assert nt > 150 and _counts(gst) == (nt, hg)
    finally:
        scene.close()
        mesh.close()
        for b in fbs + cbs:
            b.free()


def test_frame_whose_queues_hold_exactly_the_entries(ctx):
    rows = 877
    pos, idx = _grid(rows)
    mesh = crx.Mesh(ctx, pos, idx)
    view = _edge_view(rows)
    want, _, st = oracle_render(SceneSpec().add(orc.HostMesh(crx, pos, idx, None), [crx.identity()]), W, H, view,
                                wl.projection(W, H))
    t = crx.default_tuning()
    t.max_nontrivial, t.max_huge = st.num_nontrivial, st.num_huge
    scene = crx.Scene(ctx)
    scene.add(mesh)
    fb, cb = ctx.alloc(8 * W * H), ctx.alloc(8 * W * H)
    ctx.tuning = t
    try:
        frame = crx.Frame(scene, [crx.make_view(view, wl.projection(W, H), W, H)], [fb], [cb])
        for handed_out in (False, True):
            if handed_out:
                mesh.buffers()
            for _ in range(2):
                frame.launch()
                gst = frame.wait()      # raises when a queue overflows
                assert _counts(gst) == _counts(st)
                got = fb.download(np.uint64, W * H)
                assert np.array_equal(got, want), describe_mismatch(got, want, W)
        frame.close()
    finally:
        ctx.tuning = crx.default_tuning()
        scene.close()
        mesh.close()
        fb.free()
        cb.free()
