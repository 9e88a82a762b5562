"""Draws whose unit list cannot be had are drawn without one.

The list of k_cull_units is a help, not a need: a draw of more units than an
entry can name (2^31) takes the kernels that need no list and equals the walk
over all triangles (tolerance: none).
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
