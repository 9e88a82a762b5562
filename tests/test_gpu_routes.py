"""Which stage-1 kernel a draw takes (crx_context_stage1_launch).

All kernels draw the same buffers, so a draw that took another one than its
rule says would pass every comparison with the oracle.  Here are both sides of
each rule's line: few triangles per pixel and the lanes that share a triangle
there, meshes with unit boxes, several views, the tuning's knobs, and meshes
drawn over many instances.
"""
import threading
import time

import pytest

import crx
import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = crx.Context(0)
    yield c
    c.close()


@pytest.fixture(scope="module")
def large(ctx):
    """3.4 M triangles, with unit boxes."""
    mesh = crx.Mesh(ctx, *wl.heightfield_mesh(1300, amplitude=20.0, scale=200.0))
    yield mesh
    mesh.close()


def _draw(ctx, nodes, sizes, pose=((650.0, 400.0, -300.0), (650.0, 0.0, 600.0)), **tuning):
    t = crx.default_tuning()
    for k, v in tuning.items():
        setattr(t, k, v)
    ctx.tuning = t
    scene = crx.Scene(ctx)
    view = crx.look_at(*pose, (0.0, 1.0, 0.0))
    views = [crx.make_view(view, wl.projection(w, h), w, h) for w, h in sizes]
    fbs = [ctx.alloc(8 * w * h) for w, h in sizes]
    try:
        for mesh, world in nodes:
            scene.add(mesh, world)
        settings = crx.render_settings(resolve=0, frustum_culling=0)
        if len(views) == 1:
            scene.render(views[0], fbs[0], None, settings)
        else:
            scene.render_views(views, fbs, None, settings)
        return ctx.stage1_launch()
    finally:
        ctx.tuning = crx.default_tuning()
        scene.close()
        for b in fbs:
            b.free()


def test_few_triangles_per_pixel(ctx):
    mesh = crx.Mesh(ctx, *wl.sphere_mesh(50, 80))          # 8000 triangles
    pose = ((0.0, 0.3, 2.4), (0.0, 0.0, 0.0))
    assert _draw(ctx, [(mesh, None)], [(40, 50)], pose).route == crx.STAGE1_COARSE       # 4 per pixel
    assert _draw(ctx, [(mesh, None)], [(1999, 1)], pose).route == crx.STAGE1_PLAIN
    assert _draw(ctx, [(mesh, None)], [(40, 50)], pose, stage1_layout=0).route == crx.STAGE1_PLAIN
    assert _draw(ctx, [(mesh, None)], [(40, 50)] * 2, pose).route == crx.STAGE1_VIEWS
    mesh.close()


def test_lanes_that_share_a_triangle(ctx):
    """As many (up to 16) as the chip holds at once: 32 waves of 64 lanes per CU."""
    lanes = 2048 * ctx.num_cus
    for split, next_split in ((16, 8), (8, 4), (4, 2), (2, 1)):
        for triangles, want in ((lanes // split, split), (lanes // split + 2, next_split)):
            segments = next(s for s in (256, 128, 64, 32, 16, 9, 8, 7, 5, 4, 3, 2, 1) if triangles // 2 % s == 0)
            mesh = crx.Mesh(ctx, *wl.sphere_mesh(triangles // 2 // segments, segments))
            assert mesh.num_triangles == triangles
            got = _draw(ctx, [(mesh, None)], [(1000, 700)], ((0.0, 0.3, 2.4), (0.0, 0.0, 0.0)))
            mesh.close()
            assert (got.route, got.split) == (crx.STAGE1_COARSE, want), (triangles, got.split)


def test_meshes_with_boxes(ctx, large):
    one, two = [(320, 200)], [(320, 200), (200, 100)]
    assert _draw(ctx, [(large, None)], one).route == crx.STAGE1_LISTED
    assert _draw(ctx, [(large, None)], two).route == crx.STAGE1_LISTED_VIEWS
    small = crx.Mesh(ctx, *wl.heightfield_mesh(700, amplitude=20.0, scale=200.0))      # 0.98 M: without boxes
    assert _draw(ctx, [(small, None)], one).route == crx.STAGE1_PLAIN
    assert _draw(ctx, [(small, None)], two).route == crx.STAGE1_VIEWS
    assert _draw(ctx, [(small, None), (large, None)], one).route == crx.STAGE1_LISTED
    small.close()
    for knob in ({"stage1_layout": 0}, {"stage1_layout": 1}, {"stage1_block": 128}, {"stage1_strip_rows": 4},
                 {"stage1_strip_batches": 2}, {"stage1_tris_per_lane": 1}):
        assert _draw(ctx, [(large, None)], one, **knob).route == crx.STAGE1_PLAIN, knob
        assert _draw(ctx, [(large, None)], two, **knob).route == crx.STAGE1_VIEWS, knob
    # pairs over all units: enough batches for every wave of a small grid
    got = _draw(ctx, [(large, None)], one, stage1_tris_per_lane=2, stage1_waves_per_cu=4)
    assert (got.route, got.workgroups) == (crx.STAGE1_PAIRS, ctx.num_cus)


def test_handed_out_geometry(ctx):
    mesh = crx.Mesh(ctx, *wl.heightfield_mesh(1300, amplitude=20.0, scale=200.0))
    assert _draw(ctx, [(mesh, None)], [(320, 200)]).route == crx.STAGE1_LISTED
    mesh.buffers()
    assert _draw(ctx, [(mesh, None)], [(320, 200)]).route == crx.STAGE1_PLAIN
    assert _draw(ctx, [(mesh, None)], [(320, 200)] * 2).route == crx.STAGE1_VIEWS
    mesh.close()


def test_geometry_handed_out_beside_draws(ctx):
    """Another thread hands meshes out while a scene of them is drawn: once it is
    done, the next draw takes no boxes."""
    meshes = [crx.Mesh(ctx, *wl.heightfield_mesh(726, amplitude=9.0, scale=90.0)) for _ in range(6)]
    scene = crx.Scene(ctx)
    for m in meshes:
        scene.add(m)
    view = crx.make_view(crx.look_at((360.0, 200.0, -100.0), (360.0, 0.0, 300.0)), wl.projection(320, 200), 320, 200)
    fb = ctx.alloc(8 * 320 * 200)
    settings = crx.render_settings(resolve=0)

    def hand_out():
        for m in meshes:
            time.sleep(0.002)
            m.buffers()

    scene.render(view, fb, None, settings)
    assert ctx.stage1_launch().route == crx.STAGE1_LISTED
    other = threading.Thread(target=hand_out)
    other.start()
    while other.is_alive():
        scene.render(view, fb, None, settings)
    other.join()
    scene.render(view, fb, None, settings)
    assert ctx.stage1_launch().route == crx.STAGE1_PLAIN
    scene.close()
    fb.free()
    for m in meshes:
        m.close()


def test_many_instances(ctx, large):
    worlds = list(wl.instance_transforms(40, extent=60.0))
    sphere = crx.Mesh(ctx, *wl.sphere_mesh(16, 32))
    pose = ((0.0, 30.0, 150.0), (30.0, 30.0, 30.0))
    got = _draw(ctx, [(sphere, w) for w in worlds[:3]], [(320, 200)], pose)
    assert (got.route, got.shares) == (crx.STAGE1_COARSE, 1)
    got = _draw(ctx, [(sphere, w) for w in worlds[:4]], [(320, 200)], pose)
    assert (got.route, got.shares) == (crx.STAGE1_PLAIN, 1)
    got = _draw(ctx, [(sphere, w) for w in worlds], [(320, 200)], pose)
    assert (got.route, got.shares) == (crx.STAGE1_PLAIN, 10)      # shares of four instances
    assert _draw(ctx, [(sphere, w) for w in worlds], [(320, 200)] * 2, pose).route == crx.STAGE1_VIEWS
    sphere.close()


@pytest.mark.parametrize("rings,segments,count", [(500, 500, 30), (163, 625, 53), (100, 100, 40), (64, 64, 120)])
def test_shares_of_one_mesh(ctx, rings, segments, count):
    """One mesh: as many shares as its waves leave of the 28 per CU that the chip
    holds (none for a mesh that fills it), at most one per four instances."""
    mesh = crx.Mesh(ctx, *wl.sphere_mesh(rings, segments))
    worlds = wl.instance_transforms(count, extent=200.0)
    pose = ((350.0, 350.0, 350.0), (100.0, 100.0, 100.0))
    got = _draw(ctx, [(mesh, w) for w in worlds], [(800, 600)], pose)
    waves = -(-mesh.num_triangles // 64)
    want = max(1, min(int(28 * ctx.num_cus / waves + 0.5), -(-count // 4)))
    mesh.close()
    assert (got.route, got.shares) == (crx.STAGE1_PLAIN, want)


def test_shares_of_small_meshes_beside_a_large_one(ctx):
    """A mesh of few triangles of many pixels takes all its instances in a handful of
    waves, long after the large mesh is through: the draw is shared."""
    large, small = crx.Mesh(ctx, *wl.sphere_mesh(320, 320)), crx.Mesh(ctx, *wl.sphere_mesh(20, 20))
    worlds = list(wl.instance_transforms(64, extent=30.0))
    pose = ((15.0, 18.0, -12.0), (15.0, 12.0, 15.0))
    alone = _draw(ctx, [(large, w) for w in worlds[:32]], [(1365, 769)], pose)
    both = _draw(ctx, [(large, w) for w in worlds[:32]] + [(small, w) for w in worlds[32:]], [(1365, 769)], pose)
    large.close()
    small.close()
    assert alone.shares == max(1, min(8, int(28 * ctx.num_cus / 3200 + 0.5))) and both.shares > alone.shares


def test_nothing_to_draw(ctx):
    scene = crx.Scene(ctx)
    fb = ctx.alloc(8 * 64)
    scene.render(crx.make_view(crx.identity(), wl.projection(8, 8), 8, 8), fb, None, crx.render_settings(resolve=0))
    assert ctx.stage1_launch().route == crx.STAGE1_NONE
    scene.close()
    fb.free()


def test_grid_of_a_listed_draw(ctx, large):
    """stage1_waves_per_cu sets the grid of a listed draw of one float view as it does
    any other's; several views take 64 waves per CU."""
    for waves in (8, 20, 32, 64):
        got = _draw(ctx, [(large, None)], [(320, 200)], stage1_waves_per_cu=waves)
        assert got.route == crx.STAGE1_LISTED
        assert got.workgroups == min(ctx.num_cus * waves // 4, (_units(large) + 7) // 8 * 8)
    got = _draw(ctx, [(large, None)], [(320, 200)], stage1_waves_per_cu=0)         # one workgroup per unit
    assert got.workgroups == (_units(large) + 7) // 8 * 8
    for waves in (8, 32):
        got = _draw(ctx, [(large, None)], [(320, 200)] * 2, stage1_waves_per_cu=waves)
        assert got.route == crx.STAGE1_LISTED_VIEWS
        assert got.workgroups == min(ctx.num_cus * 16, (_units(large) + 7) // 8 * 8)


def _units(mesh):
    """Units of the default walk: strips of 128 triangles times groups of 8 rows, rounded up to 8."""
    row = mesh.row_triangles()
    rows = (mesh.num_triangles + row - 1) // row
    return (row + 127) // 128 * (((rows + 7) // 8 + 7) // 8 * 8)
