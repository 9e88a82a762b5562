"""Stage 1 of draws with few triangles per pixel (k_stage1_coarse).

Lane groups of 1 to 16 lanes share a triangle and draw its box rows in turn,
and a wave whose triangles lie close together takes its minima in an LDS tile
of 512 samples before it sends them to the framebuffer.  Both only change who
writes a sample and when, so the buffers must equal the oracle's bit for bit
(tolerance: none): at every number of lanes per triangle and at the triangle
counts where that number changes (524,288 lanes fill the chip), at one
triangle, at targets where the draw is just coarse (4 triangles per pixel) and
just not, at wave boxes from a few samples to wider than the tile, and for
non-indexed, IX_PU16, mirrored and near-plane draws.
"""
import numpy as np
import pytest

import crx
import oracle as orc
import workloads as wl
from crxtest import CompressedMesh, GpuScene, SceneSpec, describe_mismatch, oracle_render

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = crx.Context(0)
    yield c
    c.close()


def _check(ctx, spec, W, H, view, proj):
    want_fb, want_cb, st = oracle_render(spec, W, H, view, proj, attribute=crx.DISPLAY_VERTEX_COLORS)
    fb, cb, gst = GpuScene(ctx, spec).render(W, H, view, proj, attribute=crx.DISPLAY_VERTEX_COLORS)
    assert np.array_equal(fb, want_fb), describe_mismatch(fb, want_fb, W)
    assert np.array_equal(cb, want_cb), describe_mismatch(cb, want_cb, W)
    assert gst.num_nontrivial == st.num_nontrivial and gst.stage1_kernel == 0
    return fb


# 2 * rings * segments triangles: 16 lanes per triangle up to 32,768, 8 up to
# 65,536, 4 up to 131,072, 2 up to 262,144
@pytest.mark.parametrize("rings,segments", [(3, 4), (9, 31), (128, 128), (127, 130), (128, 256), (256, 256),
                                            (255, 258), (512, 256), (300, 437), (512, 1024)])
@pytest.mark.parametrize("W,H", [(1280, 720), (517, 1031)])
def test_lane_groups_match_the_oracle(ctx, rings, segments, W, H):
    pos, idx, col = wl.sphere_mesh(rings, segments)
    spec = SceneSpec().add(orc.HostMesh(crx, pos, idx, col), [crx.identity()])
    view = crx.look_at((0.4, 0.7, 2.1), (0.0, 0.0, 0.0), (0.2, 1.0, 0.0))
    fb = _check(ctx, spec, W, H, view, wl.projection(W, H))
    assert (fb != crx.CLEAR_PIXEL).sum() > 1000


@pytest.mark.parametrize("distance", [0.9, 1.6, 3.0, 9.0, 40.0])
def test_tile_sizes(ctx, distance):
    """A 129 x 129 grid from so near that a triangle's box exceeds the tile to
    so far that a wave's triangles share a handful of samples."""
    pos, idx, col = wl.heightfield_mesh(129, spacing=1.0 / 64, amplitude=0.05, scale=0.4)
    pos = pos - np.array([1.0, 0.0, 1.0], dtype=np.float32)
    spec = SceneSpec().add(orc.HostMesh(crx, pos, idx, col), [crx.identity()])
    view = crx.look_at((0.1, distance, -0.6 * distance), (0.0, 0.0, 0.0), (0.3, 1.0, 0.1))
    _check(ctx, spec, 1277, 719, view, wl.projection(1277, 719))


def test_one_triangle_and_the_rule_edge(ctx):
    tri = np.array([[-1, -1, 0], [1, -1, 0], [0, 1, 0]], dtype=np.float32)
    view = crx.look_at((0.0, 0.0, 30.0), (0.0, 0.0, 0.0), (0.0, 1.0, 0.0))
    spec = SceneSpec().add(orc.HostMesh(crx, tri, np.array([[0, 1, 2]], np.uint32), None), [crx.identity()])
    _check(ctx, spec, 200, 150, view, wl.projection(200, 150))
    # 2 * 50 * 80 = 8000 triangles at 40 x 50 = 2000 pixels (coarse) and at 1999 (not)
    pos, idx, col = wl.sphere_mesh(50, 80)
    spec = SceneSpec().add(orc.HostMesh(crx, pos, idx, col), [crx.identity()])
    view = crx.look_at((0.0, 0.3, 2.4), (0.0, 0.0, 0.0), (0.0, 1.0, 0.0))
    for W, H in ((40, 50), (1999, 1)):
        _check(ctx, spec, W, H, view, wl.projection(W, H))


def test_formats_mirrors_and_near_plane(ctx):
    hp, hi, hc = wl.heightfield_mesh(97, amplitude=3.0, scale=24.0)
    flat = hp[hi.reshape(-1)]
    mirror = np.diag([-1.0, 1.0, 1.0, 1.0]).astype(np.float32)
    mirror[:3, 3] = (96.0, 2.0, 40.0)
    W, H = 801, 603
    proj = wl.projection(W, H)
    views = [crx.look_at((48.0, 30.0, -30.0), (48.0, 0.0, 48.0), (0.0, 1.0, 0.0)),
             crx.look_at((48.0, 3.5, 20.0), (48.0, 1.0, 60.0), (0.0, 1.0, 0.0))]
    for mesh in (orc.HostMesh(crx, hp, hi, hc), orc.HostMesh(crx, flat, None, hc[hi.reshape(-1)]),
                 CompressedMesh(hp, hi, hc)):
        spec = SceneSpec().add(mesh, [crx.identity(), crx.Mat4.from_numpy(mirror)])
        for view in views:
            _check(ctx, spec, W, H, view, proj)
