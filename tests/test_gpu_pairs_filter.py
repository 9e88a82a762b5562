"""The filter of the pair kernel (k_stage1_pairs).

Triangles that an approximate projection proves to hold no sample never reach
the exact code; the others are gathered and drawn 64 at a time.  The filter may
only drop what the exact code neither draws nor queues, so the buffers and the
stage-2 count equal the oracle's (tolerance: none) for triangles placed on and
about sample centres, the window's edges and beyond them, from a thousandth of
a pixel to several, in both quad patterns and without shared vertices, behind
the camera, and with NaN, infinite and very large coordinates.
"""
import numpy as np
import pytest

import crx
import oracle as orc
import workloads as wl
from crxtest import SceneSpec, describe_mismatch, oracle_render

pytestmark = pytest.mark.gpu

TRIS = (1 << 20) + 1234      # past the size from which a mesh draws listed units


@pytest.fixture(scope="module")
def ctx():
    c = crx.Context(0)
    yield c
    c.close()


def _quads(count, W, H, size, seed):
    """Corners (count, 4, 3) of small quads about screen points that favour sample centres and the window's edges."""
    rng = np.random.default_rng(seed)
    pm = np.array(wl.projection(W, H).m, dtype=np.float64).reshape(4, 4)
    c = np.empty((count, 2))
    for a, n in ((0, W), (1, H)):
        any_ = rng.uniform(-2.0, n + 1.0, count)
        near = rng.choice(np.array([-2.0, -1.0, -0.5, 0.0, 1.0, n - 2.0, n - 1.0, n - 0.5, n, n + 1.0]), count)
        c[:, a] = np.where(rng.random(count) < 0.7, any_, near)
        c[:, a] = np.where(rng.random(count) < 0.3, np.round(c[:, a]), c[:, a])
    c += rng.choice(np.array([0.0, 1e-4, -1e-4, 0.01, -0.01]), (count, 2))
    e = size * 10.0 ** rng.uniform(-3.0, 0.0, (count, 1, 1))
    corners = np.array([[0.0, 0.0], [1.0, 0.0], [1.0, 1.0], [0.0, 1.0]]) - 0.5
    s = c[:, None, :] + e * (corners + rng.uniform(-0.2, 0.2, (count, 4, 2)))
    d = rng.uniform(1.0, 50.0, (count, 1, 1)) * np.ones((count, 4, 1))
    ndc = (s + 0.5) / np.array([W, H]) * 2.0 - 1.0
    return np.concatenate([ndc * d / np.array([pm[0, 0], pm[1, 1]]), -d], axis=2).astype(np.float32)


def _check(ctx, pos, idx, W, H):
    view, proj = crx.identity(), wl.projection(W, H)
    spec = SceneSpec().add(orc.HostMesh(crx, pos, idx, None), [crx.identity()])
    want, _, st = oracle_render(spec, W, H, view, proj)
    mesh = crx.Mesh(ctx, pos, idx)
    scene = crx.Scene(ctx)
    scene.add(mesh, None)
    fb, cb = ctx.alloc(8 * W * H), ctx.alloc(8 * W * H)
    try:
        gst = scene.render(crx.make_view(view, proj, W, H), fb, cb, crx.render_settings())
        got = fb.download(np.uint64, W * H)
    finally:
        fb.free()
        cb.free()
        scene.close()
        mesh.close()
    assert gst.stage1_kernel == 2 and gst.num_nontrivial == st.num_nontrivial
    assert np.array_equal(got, want), describe_mismatch(got, want, W)
    assert (got != crx.CLEAR_PIXEL).any()


PATTERNS = {"grid": (0, 1, 2, 0, 2, 3), "fan": (0, 1, 2, 0, 3, 1), "none": (0, 1, 2, 3, 0, 2)}


@pytest.mark.parametrize("pattern", sorted(PATTERNS))
@pytest.mark.parametrize("W,H,size", [(333, 217, 1.0), (333, 217, 6.0), (64, 2, 2.0), (640, 360, 0.5)])
def test_filter_matches_the_oracle(ctx, pattern, W, H, size):
    quads = _quads((TRIS + 1) // 2, W, H, size, seed=W + int(size))
    n = len(quads)
    idx = (4 * np.arange(n, dtype=np.uint32)[:, None] + np.array(PATTERNS[pattern], np.uint32)).reshape(-1, 3)[:TRIS]
    _check(ctx, quads.reshape(-1, 3), idx, W, H)


def test_special_coordinates(ctx):
    W, H = 333, 217
    quads = _quads((TRIS + 1) // 2, W, H, 3.0, seed=9)
    rng = np.random.default_rng(10)
    flat = quads.reshape(-1)
    at = rng.choice(len(flat), len(flat) // 200, replace=False)
    flat[at] = rng.choice(np.array([np.nan, np.inf, -np.inf, 0.0, -0.0, 1e30, -1e30, 3e38, 1e-30, -1e-38, 5.0], np.float32),
                          len(at))
    idx = (4 * np.arange(len(quads), dtype=np.uint32)[:, None] + np.array(PATTERNS["grid"], np.uint32)).reshape(-1, 3)
    _check(ctx, quads.reshape(-1, 3), idx[:TRIS], W, H)
