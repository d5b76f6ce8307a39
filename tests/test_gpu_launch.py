"""How launches are sized and binned: grids by what a draw can cover, whatever
its number of triangles; k_bin or the tile sort by what each draw of a frame
was in an earlier one."""
import ctypes

import numpy as np
import pytest

from conftest import plane_diffs, trace
from mytinygl_amd.gl import ENUMS as E
from test_gpu_bins import _ortho, _triangles

pytestmark = pytest.mark.gpu

ALL = E["GL_COLOR_BUFFER_BIT"] | E["GL_DEPTH_BUFFER_BIT"] | E["GL_STENCIL_BUFFER_BIT"]


@pytest.mark.parametrize("blend", [False, True])
@pytest.mark.parametrize("fb", [(8, 8), (161, 121), (640, 480), (1920, 1080), (3840, 2160)])
def test_few_triangles_get_a_whole_grid(mtgl, fb, blend):
    """A full-screen quad's raster grid fills the chip, as far as the
    framebuffer has tiles for it: two triangles say nothing of its items."""
    W, H = fb
    ctx = mtgl.create_context(W, H)
    try:
        mtgl.glViewport(0, 0, W, H)
        if blend:
            mtgl.glEnable(E["GL_BLEND"])
            mtgl.glBlendFunc(E["GL_SRC_ALPHA"], E["GL_ONE_MINUS_SRC_ALPHA"])
        mtgl.glClear(ALL)
        mtgl.glBegin(E["GL_QUADS"])
        mtgl.glColor4f(0.2, 0.4, 0.6, 0.5)
        for x, y in ((-1, -1), (1, -1), (1, 1), (-1, 1)):
            mtgl.glVertex3f(x, y, 0.5)
        mtgl.glEnd()
        mtgl.finish(ctx)
        tiles = ((W + 7) // 8) * ((H + 7) // 8)
        # four waves on each of 256 CUs, or a wave per tile where there are fewer
        assert trace(mtgl, ctx)["raster_blocks"] >= min(1024, max(1, tiles if tiles < 64 else tiles & ~63))
    finally:
        mtgl.destroy_context(ctx)
        mtgl.release()


def _frames(g, W, H, frames):
    """Draws frames of (triangles, together) draws with a wait after each;
    returns the launches of each frame by binner."""
    ctx = g.create_context(W, H)
    out = []
    try:
        _ortho(g, W, H)
        g.glEnableClientState(E["GL_VERTEX_ARRAY"])
        g.glEnableClientState(E["GL_COLOR_ARRAY"])
        for draws in frames:
            before = trace(g, ctx)
            g.glClear(ALL)
            for n, together in draws:
                pos, col = _triangles(np.random.default_rng(n), W, H, n, 9, together)
                g.glVertexPointer(3, E["GL_FLOAT"], 0, g.keep(pos))
                g.glColorPointer(4, E["GL_FLOAT"], 0, g.keep(col))
                g.glDrawArrays(E["GL_TRIANGLES"], 0, 3 * n)
            g.finish(ctx)
            after = trace(g, ctx)
            out.append((after["binned"] - before["binned"], after["sorted"] - before["sorted"]))
    finally:
        g.destroy_context(ctx)
        g.release()
    return out


MESH, SCATTERED, OVERLAY = (32_768, True), (40_000, False), (2, False)


@pytest.mark.parametrize("frame,binned,sort", [
    ([MESH], 1, 0), ([SCATTERED], 0, 1),
    ([MESH, OVERLAY], 2, 0),                # a small draw at the end says nothing of the mesh
    ([SCATTERED, OVERLAY], 1, 1),
    ([MESH, SCATTERED], 1, 1), ([SCATTERED, MESH], 1, 1),
    ([SCATTERED, MESH, OVERLAY, SCATTERED, MESH], 3, 2),
    ([(32_768, False), MESH], 1, 1),        # as many triangles: told apart by their places
], ids=lambda v: "".join("MSO"[min(d[0] == 40_000, 1) + 2 * (d[0] == 2)] for d in v) if isinstance(v, list) else None)
def test_each_draw_is_binned_by_its_own_spread(mtgl, frame, binned, sort):
    got = _frames(mtgl, 1920, 1080, [frame] * 4)
    assert got[1:] == [(binned, sort)] * 3


def test_draws_of_changing_sizes(mtgl):
    """A cloud of points that grows and shrinks from frame to frame stays sorted."""
    got = _frames(mtgl, 1920, 1080, [[(n, False)] for n in (40_000, 41_000, 38_500, 44_000, 36_000)])
    assert got[1:] == [(0, 1)] * 4


def test_more_large_draws_than_counts_are_kept_for(mtgl):
    """The counts of the latest 16 large draws of a frame reach the host."""
    n = 20
    got = _frames(mtgl, 640, 480, [[(48_000 + 64 * k, False) for k in range(n)]] * 3)
    assert got[0] == (n, 0) and got[2] == (0, n)


def _batch(g, W, H, n, rounds):
    """n contexts' (triangles, together) draws, a round each, recorded and
    launched once; the planes of each context and the rounds by binner."""
    ctxs = [g.create_context(W, H) for _ in range(n)]
    b = g.batch()
    try:
        b.begin()
        for k, c in enumerate(ctxs):
            g.gl_make_current(c)
            _ortho(g, W, H)
            g.glEnableClientState(E["GL_VERTEX_ARRAY"])
            g.glEnableClientState(E["GL_COLOR_ARRAY"])
            g.glClear(ALL)
            for m, together in rounds:
                pos, col = _triangles(np.random.default_rng(m + k), W, H, m, 9, together)
                g.glVertexPointer(3, E["GL_FLOAT"], 0, g.keep(pos))
                g.glColorPointer(4, E["GL_FLOAT"], 0, g.keep(col))
                g.glDrawArrays(E["GL_TRIANGLES"], 0, 3 * m)
        b.end(False)
        by = None
        if g.kind == "mtgl":
            fn = g.lib.mtgl_batch_launch_trace
            fn.argtypes = [ctypes.c_void_p, ctypes.POINTER(ctypes.c_uint64)]
            out = (ctypes.c_uint64 * 3)()
            assert fn(b.h, out) == 0
            by = tuple(out)
        b.launch()
        assert b.sync() == 0
        return [g.read_framebuffer(c, W, H) for c in ctxs], by
    finally:
        b.destroy()
        for c in ctxs:
            g.destroy_context(c)
        g.release()


@pytest.mark.parametrize("rounds,by", [
    ([(40_000, False)], (0, 1)), ([(32_768, True)], (1, 0)), ([(40_000, False), (32_768, True)], (1, 1)),
    ([(32_768, True), (40_000, False), (500, False)], (2, 1)),
    ([(32_768, True), (32_768, False)], (1, 1)),
], ids=["s", "m", "sm", "mso", "same"])
def test_batch_rounds_are_binned_by_their_own_spread(mtgl, oracle, rounds, by):
    """A batch learns how far its rounds' triangles lie apart while it is built."""
    W, H, n = 1024, 600, 2
    want, _ = _batch(oracle, W, H, n, rounds)
    got, took = _batch(mtgl, W, H, n, rounds)
    assert took[:2] == by
    for a, b in zip(want, got):
        assert plane_diffs(a, b) == {"color": 0, "depth": 0, "stencil": 0}


def _array(g, pos, col):
    g.glEnableClientState(E["GL_VERTEX_ARRAY"])
    g.glEnableClientState(E["GL_COLOR_ARRAY"])
    g.glVertexPointer(3, E["GL_FLOAT"], 0, g.keep(np.ascontiguousarray(pos.reshape(-1, 3), dtype=np.float32)))
    g.glColorPointer(4, E["GL_FLOAT"], 0, g.keep(np.ascontiguousarray(col, dtype=np.float32)))
    g.glDrawArrays(E["GL_TRIANGLES"], 0, pos.size // 3)


def _bars(W, H, n, upright):
    """n triangles along one edge of the screen, 16 pixels thick: one column or
    row of squares holds all their records."""
    rng = np.random.default_rng(n)
    p = np.empty((n, 3, 3))
    long_, thick = (H, 16.0) if upright else (W, 16.0)
    a = rng.uniform(0, thick, (n, 3))
    b = np.stack([np.zeros(n), np.full(n, float(long_)), rng.uniform(0, long_, n)], 1)
    p[..., 0], p[..., 1] = (a, b) if upright else (b, a)
    p[..., 2] = -rng.uniform(1.0, 90.0, (n, 1))
    return p, rng.random((3 * n, 4))


@pytest.mark.parametrize("fb,upright", [((512, 1024), True), ((480, 1024), True), ((1024, 512), False)])
def test_regions_fill_alike_and_size_only_k_bin(mtgl, oracle, fb, upright):
    """A draw whose records all lie in one column or row of squares overflows
    k_bin's room once; the room it then gets is in proportion to its records,
    and the next draw that is sorted has room for four pairs a triangle."""
    W, H = fb
    n, scattered = 3000, 80_000
    planes = []
    for g in (oracle, mtgl):
        ctx = g.create_context(W, H)
        try:
            _ortho(g, W, H)
            g.glClear(ALL)
            if g is mtgl:
                g.stats_reset(ctx)
            _array(g, *_bars(W, H, n, upright))
            planes.append(g.read_framebuffer(ctx, W, H))
            if g is mtgl:
                t = trace(g, ctx)
                pairs = g.stats(ctx).bin_pairs
                first = 32 * n + 4 * ((W + 7) // 8) * ((H + 7) // 8) + 65536
                assert pairs > first and t["reruns"] == 1 and t["sorted"] == 0
                assert pairs <= t["room"] <= 1.7 * pairs
                for _ in range(2):
                    _array(g, *_triangles(np.random.default_rng(1), W, H, scattered, 2, False))
                    g.finish(ctx)
                t = trace(g, ctx)
                assert t["sorted"] == 1 and t["room"] == 4 * scattered + 4096
        finally:
            g.destroy_context(ctx)
            g.release()
    assert plane_diffs(*planes) == {"color": 0, "depth": 0, "stencil": 0}


@pytest.mark.parametrize("fb", [(136, 72), (40, 600), (600, 40), (544, 32), (32, 544), (545, 33), (8, 8)])
def test_every_tile_heavy(mtgl, oracle, fb):
    """Eight work items for every tile: the fullest a region of the list gets,
    for rows and columns of squares around sixteen."""
    W, H = fb
    rng = np.random.default_rng(7)
    n = 260
    p = np.empty((n, 3, 3))
    p[:, 0, :2], p[:, 1, :2], p[:, 2, :2] = (-2 * W, -2 * H), (5 * W, -2 * H), (-2 * W, 5 * H)
    p[..., 2] = -rng.uniform(1.0, 90.0, (n, 3))
    col = rng.random((3 * n, 4))
    planes = []
    for g in (oracle, mtgl):
        ctx = g.create_context(W, H)
        try:
            _ortho(g, W, H)
            g.glEnable(E["GL_BLEND"])
            g.glBlendFunc(E["GL_SRC_ALPHA"], E["GL_ONE_MINUS_SRC_ALPHA"])
            g.glClear(ALL)
            _array(g, p, col)
            planes.append(g.read_framebuffer(ctx, W, H))
            if g is mtgl:
                assert trace(g, ctx)["binned"] >= 1
        finally:
            g.destroy_context(ctx)
            g.release()
    assert plane_diffs(*planes) == {"color": 0, "depth": 0, "stencil": 0}


def test_sorted_draw_of_several_vertex_states(mtgl, oracle):
    """A draw whose material changes between vertices, binned and then sorted
    (set-up's variants that read the states from memory), lit, scattered, and
    with triangles past the near and far planes."""
    W, H, n = 1920, 1080, 7_000
    pos, col = _triangles(np.random.default_rng(5), W, H, n, 9, False)
    pos, col = pos.tolist(), col.tolist()
    out = []
    for g in (oracle, mtgl):
        ctx = g.create_context(W, H)
        try:
            _ortho(g, W, H)
            g.glEnable(E["GL_LIGHTING"])
            g.glEnable(E["GL_LIGHT0"])
            g.glNormal3f(0.0, 0.0, 1.0)
            for _ in range(2):
                g.glClear(ALL)
                g.glBegin(E["GL_TRIANGLES"])
                for k, (p, c) in enumerate(zip(pos, col)):
                    if k % 1000 == 1:
                        g.glMaterialfv(E["GL_FRONT_AND_BACK"], E["GL_DIFFUSE"], g.fv(*c))
                    g.glVertex3f(*p)
                g.glEnd()
                out.append(g.read_framebuffer(ctx, W, H))
            if g is mtgl:
                t = trace(g, ctx)
                assert t["binned"] >= 1 and t["sorted"] >= 1
        finally:
            g.destroy_context(ctx)
            g.release()
    for a, b in zip(out[:2], out[2:]):
        assert plane_diffs(a, b) == {"color": 0, "depth": 0, "stencil": 0}
    assert (out[0][0] != out[0][0][0, 0]).sum() > W * H // 50
