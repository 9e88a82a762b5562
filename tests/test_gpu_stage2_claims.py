"""Stage-2 claims and the clipped bounding boxes (k_stage2).

A wave's claim takes entries a whole round of claims apart, and later claims
come from a cursor; a lane clips its triangle in the wave's LDS.  Neither may
change a result: the visibility buffer equals the oracle's bit for bit
(tolerance: none) at one entry, at claims of one and of several entries, at
the last claim of the static round and past it (a grid of 4 waves per CU
reaches the cursor at 65,536 entries), for triangles inside the window, across
each of its edges and corners, and across the near plane.
"""
import numpy as np
import pytest

import crx
import oracle as orc
import workloads as wl
from crxtest import GpuScene, SceneSpec, describe_mismatch, oracle_render

pytestmark = pytest.mark.gpu

W, H = 401, 303


@pytest.fixture(scope="module")
def ctx():
    c = crx.Context(0)
    yield c
    c.close()


def _soup(count, lo, hi, behind, seed):
    """Triangles `lo` to `hi` pixels wide about points in and around the window, a share `behind` of their vertices
    behind the camera (camera at the origin, looking along -z)."""
    rng = np.random.default_rng(seed)
    proj = wl.projection(W, H)
    pm = np.array(proj.m, dtype=np.float64).reshape(4, 4)
    c = rng.uniform(-0.15, 1.15, (count, 1, 2))
    s = c + rng.uniform(-0.5, 0.5, (count, 3, 2)) * rng.uniform(lo, hi, (count, 1, 1)) / np.array([W, H])
    d = rng.uniform(2.0, 40.0, (count, 3, 1)) * np.ones((count, 3, 1))
    xy = (2.0 * s - 1.0) * d / np.array([pm[0, 0], pm[1, 1]])
    z = np.where(rng.random((count, 3, 1)) < behind, rng.uniform(-1.0, 3.0, (count, 3, 1)), -d)
    pos = np.concatenate([xy, z], axis=2).astype(np.float32).reshape(-1, 3)
    return pos, np.arange(3 * count, dtype=np.uint32).reshape(-1, 3), proj


@pytest.mark.parametrize("count,lo,hi,behind,waves", [(1, 30, 60, 0.0, 16), (65, 30, 80, 0.1, 16),
                                                      (5000, 20, 70, 0.02, 16), (70001, 18, 40, 0.0, 4),
                                                      (140000, 18, 30, 0.01, 4)])
def test_claims_match_the_oracle(ctx, count, lo, hi, behind, waves):
    pos, idx, proj = _soup(count, lo, hi, behind, seed=count)
    spec = SceneSpec().add(orc.HostMesh(crx, pos, idx, None), [crx.identity()])
    view = crx.identity()
    want, _, st = oracle_render(spec, W, H, view, proj)
    tuning = crx.default_tuning()
    tuning.stage2_waves_per_cu = waves
    ctx.tuning = tuning
    try:
        got, _, gst = GpuScene(ctx, spec).render(W, H, view, proj)
    finally:
        ctx.tuning = crx.default_tuning()
    assert gst.num_nontrivial == st.num_nontrivial and gst.num_huge == st.num_huge
    assert np.array_equal(got, want), describe_mismatch(got, want, W)
