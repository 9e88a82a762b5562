"""Meshes drawn over many instances: shares, filter and pair queue (k_stage1).

Workgroups share a batch's instances, a share of few instances takes no box
tests, and the (triangle, instance) pairs that the filter leaves are drawn 64
at a time.  The visibility buffer equals the oracle's bit for bit (tolerance:
none) at the instance counts where the shares, the 64-instance lists and the box
tests change, for meshes of less than a wave to many batches, with instances
mirrored, at the near plane, behind the camera and off the window.
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


@pytest.mark.parametrize("count", [4, 8, 9, 33, 64, 65, 130, 700])
@pytest.mark.parametrize("rings,segments,compressed", [(3, 5, False), (40, 61, False), (40, 61, True), (300, 301, False)])
def test_counts_match_the_oracle(ctx, count, rings, segments, compressed):
    pos, idx, _ = wl.sphere_mesh(rings, segments, seed=rings)
    worlds = list(wl.instance_transforms(count, extent=24.0, seed=count))
    for k, w in enumerate(worlds):
        if k % 5 == 2:
            for e in range(4):
                w.m[e] = -w.m[e]
    mesh = CompressedMesh(pos, idx) if compressed else orc.HostMesh(crx, pos, idx, None)
    sp, si, _ = wl.sphere_mesh(7, 9)
    small = CompressedMesh(sp, si) if compressed else orc.HostMesh(crx, sp, si, None)
    spec = SceneSpec().add(mesh, worlds).add(small, worlds[:2])
    W, H = 357, 241
    proj = wl.projection(W, H)
    for eye, at in (((12.0, 12.0, 12.5), (20.0, 12.0, 0.0)), ((60.0, 70.0, 80.0), (12.0, 12.0, 12.0))):
        view = crx.look_at(eye, at, (0.0, 1.0, 0.0))
        want, _, st = oracle_render(spec, W, H, view, proj)
        got, _, gst = GpuScene(ctx, spec).render(W, H, view, proj)
        assert np.array_equal(got, want), describe_mismatch(got, want, W)
        assert gst.num_nontrivial == st.num_nontrivial
