"""The stage-1 filter (filter_culls) on single non-finite view coordinates.

The filter may only drop what the exact code neither draws nor queues.  A
finite vertex under a finite matrix can have a NaN in one view row (inf - inf)
with a finite depth; a minimum that skips the NaN would put the triangle off
the side where its other two vertices lie, while the exact frustum test, which
needs all three, keeps it.  Buffers and stage-2 counts equal the oracle's
(tolerance: none).
"""
import numpy as np
import pytest

import crx
import oracle as orc
import workloads as wl
from crxtest import GpuScene, SceneSpec, describe_mismatch, oracle_render

pytestmark = pytest.mark.gpu

TRIS = (1 << 20) + 100      # past the size from which a mesh draws listed units


@pytest.fixture(scope="module")
def ctx():
    c = crx.Context(0)
    yield c
    c.close()


def _world(axis):
    """View row `axis` is 10 * px - 10 * py, the other one pz; the depth is 5."""
    m = np.zeros((4, 4), dtype=np.float32)
    m[axis, 0], m[axis, 1] = 10.0, -10.0
    m[1 - axis, 2] = 1.0
    m[2, 3], m[3, 3] = -5.0, 1.0
    return crx.Mat4.from_numpy(m)


def _one_nan(axis_value, count):
    """count triangles, one vertex of each (in turn) with the NaN, the others at axis_value."""
    t = np.arange(count)
    p = np.zeros((count, 3, 3), dtype=np.float32)
    p[:, :, 0] = axis_value + np.arange(3, dtype=np.float32)
    p[:, :, 2] = np.array([-0.1, 0.3, 0.2], dtype=np.float32)
    p[t, t % 3, 0] = p[t, t % 3, 1] = 3e38
    return p.reshape(-1, 3)


def _listed(ctx, pos, idx, world, W, H, view, proj):
    mesh, scene = crx.Mesh(ctx, pos, idx), crx.Scene(ctx)
    scene.add(mesh, world)
    fb = ctx.alloc(8 * W * H)
    try:
        st = scene.render(crx.make_view(view, proj, W, H), fb, None,
                          crx.render_settings(resolve=0, frustum_culling=0))
        assert st.stage1_kernel == 2
        return fb.download(np.uint64, W * H), st
    finally:
        fb.free()
        scene.close()
        mesh.close()


@pytest.mark.parametrize("side", [-50.0, 50.0])
@pytest.mark.parametrize("axis", [0, 1])
def test_nan_in_one_view_row_of_one_vertex(ctx, axis, side):
    W, H = 333, 217
    proj = wl.projection(W, H)
    # drawn over instances (the filter of k_stage1)
    pos = _one_nan(side, 12)
    idx = np.arange(36, dtype=np.uint32).reshape(-1, 3)
    spec = SceneSpec().add(orc.HostMesh(crx, pos, idx, None), [_world(axis)] * 5)
    want, _, st = oracle_render(spec, W, H, crx.identity(), proj)
    assert st.num_nontrivial == (60 if side < 0.0 else 0)
    fb, _, gst = GpuScene(ctx, spec).render(W, H, crx.identity(), proj)
    assert np.array_equal(fb, want), describe_mismatch(fb, want, W)
    assert (gst.num_nontrivial, gst.num_huge) == (st.num_nontrivial, st.num_huge)
    # one instance of a mesh with boxes (the filter of k_stage1_pairs)
    many = np.concatenate([pos, np.tile(np.array([[0, 0, 9]], dtype=np.float32), (3 * (TRIS - 12), 1))])
    idx = np.arange(3 * TRIS, dtype=np.uint32).reshape(-1, 3)
    spec = SceneSpec().add(orc.HostMesh(crx, many, idx, None), [_world(axis)])
    want, _, st = oracle_render(spec, W, H, crx.identity(), proj)
    assert st.num_nontrivial == (12 if side < 0.0 else 0)
    fb, gst = _listed(ctx, many, idx, _world(axis), W, H, crx.identity(), proj)
    assert np.array_equal(fb, want), describe_mismatch(fb, want, W)
    assert (gst.num_nontrivial, gst.num_huge) == (st.num_nontrivial, st.num_huge)
