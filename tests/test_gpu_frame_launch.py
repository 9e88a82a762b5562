"""A launch of a recorded frame draws the records of its last crx_frame_set_views.

The frame's draw items carry the boxes of their meshes' units.  Once
crx_mesh_buffers hands a mesh's geometry out, those boxes no longer count, and
the next launch must draw without them.  Nothing else of the scene or of the
tuning reaches a launch: it neither refuses nor takes up what changed since.
Every launch must equal the walk over all triangles (tolerance: none).
"""
import ctypes as C

import numpy as np
import pytest

import crx
import workloads as wl
from crxtest import describe_mismatch

pytestmark = pytest.mark.gpu

N = 801     # 1.28 M triangles, past the size from which a mesh has boxes
W, H = 500, 300


@pytest.fixture(scope="module")
def ctx():
    c = crx.Context(0)
    yield c
    c.close()


@pytest.fixture(scope="module")
def terrain():
    return wl.heightfield_mesh(N, amplitude=20.0, scale=100.0)


def _view(dx=0.0):
    c = 0.5 * (N - 1)
    v = crx.look_at((c + dx, 60.0, -40.0), (c, 30.0, 0.0), (0.0, 1.0, 0.0))
    return crx.make_view(v, wl.projection(W, H), W, H)


class _Rig:
    """A scene of one terrain, and buffers for a frame and for plain draws."""

    def __init__(self, ctx, terrain):
        self.ctx, self.mesh, self.scene = ctx, crx.Mesh(ctx, *terrain), crx.Scene(ctx)
        self.node = self.scene.add(self.mesh)
        self.bufs = [ctx.alloc(8 * W * H) for _ in range(4)]
        self.frames = []

    def frame(self, view):
        self.frames.append(crx.Frame(self.scene, [view], self.bufs[:1], self.bufs[1:2]))
        return self.frames[-1]

    def launched(self, frame):
        frame.launch()
        frame.wait()
        return [b.download(np.uint64, W * H) for b in self.bufs[:2]]

    def whole_walk(self, view):
        t = crx.default_tuning()
        t.stage1_layout = 0
        self.ctx.tuning = t
        try:
            self.scene.render(view, self.bufs[2], self.bufs[3], crx.render_settings())
            return [b.download(np.uint64, W * H) for b in self.bufs[2:]]
        finally:
            self.ctx.tuning = crx.default_tuning()

    def move(self, pos):
        """Hands the geometry out and turns it half round its vertical axis: the far
        rows, which the view saw nothing of, come to lie before the camera."""
        p, _, _ = self.mesh.buffers()
        moved = np.ascontiguousarray(pos * np.array([-1, 1, -1], np.float32) + np.array([N - 1, 0, N - 1], np.float32))
        crx._check(crx.lib().crx_memcpy_htod(self.ctx.handle, C.c_void_p(p), C.c_void_p(moved.ctypes.data),
                                             moved.nbytes, None))

    def close(self):
        for f in self.frames:
            f.close()
        self.scene.close()
        self.mesh.close()
        for b in self.bufs:
            b.free()


@pytest.fixture
def rig(ctx, terrain):
    r = _Rig(ctx, terrain)
    yield r
    r.close()


def _same(got, want):
    for a, b in zip(got, want):
        assert np.array_equal(a, b), describe_mismatch(a, b, W)


@pytest.mark.parametrize("refused", ["nothing", "launch under another layout", "set_views after add_node"])
def test_moved_geometry(rig, terrain, refused):
    """The vertices move after the frame was recorded: every later launch
    draws the moved ones, also after a call on the frame was refused."""
    f = rig.frame(_view())
    first = rig.launched(f)
    _same(first, rig.whole_walk(_view()))
    rig.move(terrain[0])
    want = rig.whole_walk(_view())
    assert not np.array_equal(first[0], want[0])
    if refused == "launch under another layout":
        t = crx.default_tuning()
        t.stage1_layout = 0
        rig.ctx.tuning = t
        try:
            _same(rig.launched(f), want)
        finally:
            rig.ctx.tuning = crx.default_tuning()
    elif refused == "set_views after add_node":
        rig.scene.add(rig.mesh)
        with pytest.raises(crx.CrxError):
            f.set_views([_view(5.0)])
    for _ in range(2):
        _same(rig.launched(f), want)


@pytest.mark.parametrize("trigger", ["set_attributes", "buffers"])
def test_launch_repeats_the_recorded_scene(rig, terrain, trigger):
    """A node added, a node moved and the tuning changed after the recording,
    and then an attribute set or the geometry handed out (unchanged): the
    launch still draws the recorded frame."""
    f = rig.frame(_view())
    first = rig.launched(f)
    rig.scene.set_transform(rig.node, crx.Mat4.from_numpy(np.array(
        [[1, 0, 0, 40], [0, 1, 0, -20], [0, 0, 1, 10], [0, 0, 0, 1]], dtype=np.float32)))
    if trigger == "set_attributes":
        rig.mesh.set_attributes(uvs=np.zeros((len(terrain[0]), 2), dtype=np.float32))
    else:
        rig.mesh.buffers()
    _same(rig.launched(f), first)
    rig.scene.add(rig.mesh)
    _same(rig.launched(f), first)
    t = crx.default_tuning()
    t.stage1_layout = 0
    rig.ctx.tuning = t
    try:
        _same(rig.launched(f), first)
    finally:
        rig.ctx.tuning = crx.default_tuning()


def test_set_views_takes_up_transforms(rig):
    """set_views draws the scene's transforms of that moment."""
    f = rig.frame(_view())
    rig.launched(f)
    rig.scene.set_transform(rig.node, crx.Mat4.from_numpy(np.array(
        [[1, 0, 0, 15], [0, 1, 0, -8], [0, 0, 1, 10], [0, 0, 0, 1]], dtype=np.float32)))
    rig.mesh.buffers()
    f.set_views([_view(5.0)])
    _same(rig.launched(f), rig.whole_walk(_view(5.0)))


def test_frame_on_another_context(rig, terrain):
    """A frame recorded on one context over another context's scene."""
    other = crx.Context(0)
    view = _view()
    try:
        h = C.c_void_p()
        arr = (crx.View * 1)(view)
        s = crx.render_settings()
        crx._check(crx.lib().crx_frame_create(other.handle, rig.scene.handle, arr, 1, C.byref(s),
                                              (C.c_void_p * 1)(rig.bufs[0].ptr), (C.c_void_p * 1)(rig.bufs[1].ptr),
                                              C.byref(h)))
        f = crx.Frame.__new__(crx.Frame)
        f.n, f.handle = 1, h.value
        try:
            _same(rig.launched(f), rig.whole_walk(view))
            rig.move(terrain[0])
            _same(rig.launched(f), rig.whole_walk(view))
        finally:
            f.close()
    finally:
        other.close()
