"""Draws whose unit list cannot be had are drawn without one.

The list of k_cull_units is a help, not a need: when its memory cannot be
allocated, or the draw has more units than an entry can name (2^31), the draw
takes the kernels that need no list and equals the walk over all triangles
(tolerance: none).
"""
import numpy as np
import pytest

import crx
import workloads as wl
from crxtest import describe_mismatch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = crx.Context(0)
    yield c
    c.close()


ROWS, COLS, UNITS = 8, 1 << 16, 8192


def _long_rows(ctx):
    """Eight rows of 2^16 quads, 8192 units (a strip's groups of rows are rounded up to eight)."""
    z, x = np.meshgrid(np.arange(ROWS + 1, dtype=np.float32), np.arange(COLS + 1, dtype=np.float32), indexing="ij")
    pos = np.stack([x - 0.5 * COLS, 0.2 * np.sin(x), z], axis=2).reshape(-1, 3).astype(np.float32)
    a = (np.arange(ROWS, dtype=np.uint32)[:, None] * np.uint32(COLS + 1) + np.arange(COLS, dtype=np.uint32)).reshape(-1)
    b, c, d = a + np.uint32(1), a + np.uint32(COLS + 1), a + np.uint32(COLS + 2)
    mesh = crx.Mesh(ctx, pos, np.stack([a, c, d, a, d, b], axis=1).reshape(-1, 3))
    assert mesh.row_triangles() == 2 * COLS
    return mesh


def _fill(ctx, leave):
    """Takes the device's memory until an allocation of `leave` bytes fails."""
    held, size = [], 1 << 34
    while size >= leave:
        try:
            held.append(ctx.alloc(size))
        except crx.CrxError:
            size >>= 1
    return held


def test_no_memory_for_the_list():
    """16 nodes of 8192 units in 256 views: a list of 256 MB, of which the device
    has 128 to 160 MB left."""
    nodes, views, side = 16, 256, 24
    c = crx.Context(0)      # its buffers hold nothing of an earlier draw's list
    mesh = scene = None
    held, bufs = [], []
    try:
        mesh, scene = _long_rows(c), crx.Scene(c)
        for k in range(nodes):
            w = np.eye(4, dtype=np.float32)
            w[2, 3] = 10.0 * k
            scene.add(mesh, crx.Mat4.from_numpy(w))
        vs = [crx.make_view(crx.look_at((40.0 * k - 5000.0, 30.0, -9.0), (40.0 * k - 5000.0, 0.0, 40.0), (0.0, 1.0, 0.0)),
                            wl.projection(side, side), side, side) for k in range(views)]
        bufs = [c.alloc(8 * side * side) for _ in vs]
        settings = crx.render_settings(resolve=0, instanced=0, frustum_culling=0)

        def draw(layout):
            t = crx.default_tuning()
            t.stage1_layout = layout
            c.tuning = t
            st = scene.render_views(vs, bufs, None, settings)
            return st.stage1_kernel, [b.download(np.uint64, side * side) for b in bufs]

        kernel, want = draw(0)              # all other buffers of a draw are in place
        assert sum((w != crx.CLEAR_PIXEL).any() for w in want) > views // 2
        assert kernel == 1
        room = c.alloc(128 << 20)
        held = _fill(c, 32 << 20)
        room.free()
        with pytest.raises(crx.CrxError):
            c.alloc(8 * nodes * UNITS * views)
        crx.lib().hipGetLastError()         # the failed allocations' error is not the draw's
        kernel, got = draw(2)
        assert kernel == 1
        for k in range(views):
            assert np.array_equal(got[k], want[k]), describe_mismatch(got[k], want[k], side)
        for b in held:
            b.free()
        held = []
        kernel, got = draw(2)               # with the memory back, from the list
        assert kernel == 2
        for k in range(views):
            assert np.array_equal(got[k], want[k]), describe_mismatch(got[k], want[k], side)
    finally:
        for b in held + bufs:
            b.free()
        if scene is not None:
            scene.close()
        if mesh is not None:
            mesh.close()
        c.close()


@pytest.mark.parametrize("frame", [False, True])
def test_more_units_than_entries_can_name(ctx, frame):
    """2^18 nodes of 8192 units."""
    nodes = (1 << 31) // UNITS
    mesh = _long_rows(ctx)
    scene = crx.Scene(ctx)
    W, H = 64, 32
    view = crx.make_view(crx.look_at((0.0, 2.0, -3.0), (0.0, 0.0, 1.0), (0.0, 1.0, 0.0)), wl.projection(W, H), W, H)
    settings = crx.render_settings(resolve=0, instanced=0, frustum_culling=0)
    fb = ctx.alloc(8 * W * H)
    try:
        scene.add(mesh)
        scene.render(view, fb, None, settings)
        want = fb.download(np.uint64, W * H)
        assert (want != crx.CLEAR_PIXEL).any()
        # the other nodes lie behind the camera
        far = np.eye(4, dtype=np.float32)
        far[2, 3] = -1000.0
        far = crx.Mat4.from_numpy(far)
        for _ in range(nodes - 1):
            scene.add(mesh, far)
        if frame:
            f = crx.Frame(scene, [view], [fb], None, settings)
            f.launch()
            f.wait()
            f.close()
        else:
            st = scene.render(view, fb, None, settings)
            assert st.num_triangles == nodes * mesh.num_triangles
        got = fb.download(np.uint64, W * H)
        assert np.array_equal(got, want), describe_mismatch(got, want, W)
    finally:
        fb.free()
        scene.close()
        mesh.close()


def test_mesh_after_a_failed_allocation(ctx):
    """An allocation that failed leaves its error behind in the runtime; a mesh made
    next, whose boxes take a launch, is none the worse for it."""
    with pytest.raises(crx.CrxError):
        ctx.alloc(1 << 50)
    mesh = _long_rows(ctx)
    mesh.close()
