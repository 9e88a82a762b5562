"""Unit boxes of the server's nodes.

The server computes the boxes of a node's units after each upload into the
node's cache slot, in the layout of the row length that it found in the node's
index order, and draws of 2^20 triangles and more skip the units no view sees.
Nodes of different row lengths (long rows, rows too short for strips, no index
buffer, shuffled) share slots, so a slot's boxes change their layout with
every eviction; a view of more nodes than the cache holds is drawn in groups.
Every result equals the oracle's draw of the nodes the view sees (tolerance:
none).
"""
import ctypes
import time

import numpy as np
import pytest

import crx
import oracle as orc
import workloads as wl
from crxtest import describe_mismatch

pytestmark = pytest.mark.gpu

SIDE = 600.0


@pytest.fixture(scope="module")
def ctx():
    c = crx.Context(0)
    yield c
    c.close()


def _node(ctx, kind, rows, cols, x0, z0, seed):
    """A SIDE x SIDE patch at (x0, z0) as rows x cols quads in page-locked memory."""
    z, x = np.meshgrid(np.linspace(0.0, SIDE, rows + 1), np.linspace(0.0, SIDE, cols + 1), indexing="ij")
    y = 6.0 * np.sin((x + x0) / 37.0) * np.cos((z + z0) / 51.0)
    pos = np.stack([x + x0, y, z + z0], axis=2).reshape(-1, 3).astype(np.float32)
    a = (np.arange(rows, dtype=np.uint32)[:, None] * np.uint32(cols + 1) + np.arange(cols, dtype=np.uint32)).reshape(-1)
    b, c, d = a + np.uint32(1), a + np.uint32(cols + 1), a + np.uint32(cols + 2)
    idx = np.stack([a, c, d, a, d, b], axis=1).reshape(-1, 3)
    rng = np.random.default_rng(seed)
    if kind == "shuffled":
        idx = idx[rng.permutation(len(idx))]
    if kind == "plain":
        pos, idx = pos[idx.reshape(-1)], None
    col = rng.integers(0, 1 << 32, len(pos), dtype=np.uint32)
    nt = 2 * rows * cols
    buf = crx.PinnedBuffer(ctx, pos.nbytes + col.nbytes + (idx.nbytes if idx is not None else 0))
    buf.array(np.float32, pos.size)[:] = pos.reshape(-1)
    buf.array(np.uint32, col.size, pos.nbytes)[:] = col
    if idx is not None:
        buf.array(np.uint32, idx.size, pos.nbytes + col.nbytes)[:] = idx.reshape(-1)
    lo, hi = pos.min(axis=0), pos.max(axis=0)
    return buf, {"pos": buf.ptr, "col": buf.ptr + pos.nbytes,
                 "idx": buf.ptr + pos.nbytes + col.nbytes if idx is not None else None, "nv": len(pos), "nt": nt,
                 "aabb": crx.Box3(crx.Vec3(*map(float, lo)), crx.Vec3(*map(float, hi)))}


# 1.69 to 1.72 M triangles each: two of them are enough for a draw that culls its units
KINDS = [("rows", 920, 930), ("rows", 460, 1840), ("rows", 1840, 461), ("shuffled", 800, 1060), ("plain", 920, 922),
         ("rows", 921, 925)]


@pytest.fixture(scope="module")
def nodes(ctx):
    made = [_node(ctx, k, r, c, SIDE * (i % 3), SIDE * (i // 3), i) for i, (k, r, c) in enumerate(KINDS)]
    yield [n for _, n in made]
    for b, _ in made:
        b.free()


def _server(ctx, nodes, slots, batch, lanes, frame_mb=16):
    al = lambda x: (x + 255) // 256 * 256
    slot = max(al(n["nv"] * 12) + al(n["nt"] * 12) + al(n["nv"] * 4) for n in nodes)
    cfg = crx.server_config(node_cache_bytes=slot * slots, frame_bytes=frame_mb << 20, max_batch_views=batch,
                            lanes=lanes, resolve=1)
    srv = crx.Server(ctx, cfg)
    for nd in nodes:
        srv.add_node(nd["pos"], nd["nv"], nd["idx"], nd["nt"], nd["col"], nd["aabb"])
    srv.start()
    assert srv.stats().cache_slots == slots
    return srv


def _oracle_view(nodes, ids, v):
    prefix = np.concatenate([[0], np.cumsum([nd["nt"] for nd in nodes])[:-1]]).astype(np.uint64)
    inst = []
    for j, i in enumerate(ids):
        nd = nodes[i]
        m = crx.CMesh()
        m.numTriangles, m.numVertices, m.isLoaded, m.id = nd["nt"], nd["nv"], 1, i
        m.positions, m.indices, m.colors = nd["pos"], nd["idx"], nd["col"]
        m.cummulativeTriangleCount = int(prefix[i])
        m.instances.offset, m.instances.count = j, 1
        m.world = crx.identity()
        inst.append(m)
    xf = [crx.mat4_mul(v.view, crx.identity()) for _ in ids]
    fb, _ = orc.draw(crx, inst, inst, xf, v.width, v.height, v.view, v.proj, False)
    cb = orc.resolve(crx, inst, prefix[ids], fb, v.width, v.height, v.view, v.proj, crx.DISPLAY_VERTEX_COLORS)
    return fb, cb


def _views():
    """Each sees two to four nodes, part of each, from low over the ground."""
    up = (0.0, 1.0, 0.0)
    eyes = [((300.0, 40.0, -60.0), (320.0, 0.0, 300.0)), ((1500.0, 30.0, 1260.0), (1480.0, 0.0, 900.0)),
            ((-50.0, 60.0, 500.0), (500.0, 0.0, 620.0)), ((1850.0, 50.0, 640.0), (1300.0, 0.0, 560.0)),
            ((590.0, 12.0, 610.0), (900.0, 0.0, 300.0)), ((900.0, 25.0, 610.0), (880.0, 0.0, 900.0))]
    sizes = [(320, 240), (200, 150), (256, 144), (97, 131), (320, 200), (160, 160)]
    return [crx.make_view(crx.look_at(e, a, up), wl.projection(w, h), w, h) for (e, a), (w, h) in zip(eyes, sizes)]


def _fetch(srv, ticket, v):
    r = srv.wait(ticket)
    assert r.status == 0, crx.lib().crx_last_error()
    n = v.width * v.height
    out = srv.download(r.framebuffer, n), srv.download(r.colorbuffer, n)
    srv.release(ticket)
    return out


def _same(got, want, v, what):
    assert np.array_equal(got[0], want[0]), what + "\n" + describe_mismatch(got[0], want[0], v.width)
    assert np.array_equal(got[1], want[1]), what + " colours"


@pytest.mark.parametrize("slots,batch,lanes", [(6, 1, 1), (4, 1, 1), (4, 6, 2), (2, 4, 2)])
def test_results_equal_the_oracle(ctx, nodes, slots, batch, lanes):
    views = _views()
    srv = _server(ctx, nodes, slots, batch, lanes)
    try:
        ids = [srv.view_nodes(v) for v in views]
        assert all(sum(nodes[i]["nt"] for i in k) > 3 << 20 for k in ids) and any(len(k) > 4 for k in ids)
        want = [_oracle_view(nodes, k, v) for k, v in zip(ids, views)]
        for _ in range(2):                                    # the second round finds other nodes in the slots
            for k, v in enumerate(views):
                _same(_fetch(srv, srv.submit(v), v), want[k], v, f"request {k} alone")
                if lanes == 1:
                    assert srv.stage1_launch(0).route == crx.STAGE1_LISTED
        tickets = [srv.submit(v) for v in views]              # all at once
        for k, (t, v) in enumerate(zip(tickets, views)):
            _same(_fetch(srv, t, v), want[k], v, f"request {k} in a batch")
        routes = {srv.stage1_launch(l).route for l in range(lanes)} - {crx.STAGE1_NONE}
        assert routes <= {crx.STAGE1_LISTED, crx.STAGE1_LISTED_VIEWS}
        st = srv.stats()
        assert st.evictions > 0 or slots == len(nodes)
        print(f"[server] slots {slots}: uploads {st.uploads} evictions {st.evictions} max batch {st.max_batch}", flush=True)
    finally:
        srv.close()


def test_start_does_not_search_every_node(ctx):
    """1000 nodes of 8192 triangles start about as fast with an index buffer each, of
    the same or of alternating content, as with one for all: the search for a
    node's row length may take 0.1 ms (hash maps over the window took 0.25 and more)."""
    count = 1000
    kinds = [_node(ctx, "rows", r, c, 0.0, 0.0, 1) for r, c in ((64, 64), (32, 128))]
    words = 3 * 8192
    copies = crx.PinnedBuffer(ctx, 4 * words * count)
    idx = copies.array(np.uint32, words * count).reshape(count, words)
    try:
        nodes = [n for _, n in kinds]
        took = {}
        for name in ("shared", "copies", "alternating"):
            for k in range(count):
                nd = nodes[k % 2 if name == "alternating" else 0]
                idx[k] = np.ctypeslib.as_array((ctypes.c_uint32 * words).from_address(nd["idx"]))
            best = 1e9
            for _ in range(4):
                srv = crx.Server(ctx, crx.server_config(node_cache_bytes=16 << 20, frame_bytes=1 << 20,
                                                        max_batch_views=4, lanes=1, resolve=0, prefetch=0))
                for k in range(count):
                    nd = nodes[k % 2 if name == "alternating" else 0]
                    at = nd["idx"] if name == "shared" else copies.ptr + 4 * words * k
                    srv.add_node(nd["pos"], nd["nv"], at, nd["nt"], nd["col"], nd["aabb"])
                t0 = time.perf_counter()
                srv.start()
                best = min(best, time.perf_counter() - t0)
                srv.close()
            took[name] = best
        print("[server] start of 1000 nodes:", {k: f"{1e3 * v:.1f} ms" for k, v in took.items()}, flush=True)
        assert took["copies"] < took["shared"] + 1e-4 * count
        assert took["alternating"] < took["shared"] + 1e-4 * count
    finally:
        copies.free()
        for b, _ in kinds:
            b.free()
