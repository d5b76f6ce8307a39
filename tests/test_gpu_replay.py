"""Draws that overflow the device's arrays run again, in order.

The device queues draws without waiting for them.  It sizes the arrays of a
launch's (tile, triangle) pairs from its triangles and tiles and what earlier
launches needed, and the clip pool from earlier clipped triangles; a launch
that needs more poisons the context's stream (its raster stage and every later
framebuffer write are skipped), and the next call that waits for the stream
grows the arrays and runs the logged clears and draws again from that launch
on.  These frames make launches of a fresh context overflow all three ways
(the room of k_bin's regions, the tile sort's pairs, the clip pool), between
other clears and draws, and must equal the oracle's frames."""
import ctypes as C

import numpy as np
import pytest

from conftest import color_histogram, plane_diffs, trace
from mytinygl_amd import diff as D
from mytinygl_amd import scenes as S
from mytinygl_amd.gl import ENUMS as E
from test_gpu_bins import _ortho, _triangles
from test_gpu_launch import _array

pytestmark = pytest.mark.gpu


def _big_triangles(g, rng, n, W, H):
    """n triangles of about a third of the screen each: tens of bins per triangle."""
    g.glBegin(E["GL_TRIANGLES"])
    for _ in range(n):
        c = rng.uniform(0, 1, 2)
        for k in range(3):
            g.glColor4f(*rng.random(4).astype(np.float32))
            p = c + rng.uniform(-0.45, 0.45, 2)
            g.glVertex3f(float(p[0] * W), float(p[1] * H), float(-rng.uniform(0.2, 50.0)))
    g.glEnd()


def _near_plane_fan(g, rng, n):
    """n triangles crossing the near plane (each clipped into up to 2 fan triangles)."""
    g.glBegin(E["GL_TRIANGLES"])
    for _ in range(n):
        for k in range(3):
            g.glColor4f(*rng.random(4).astype(np.float32))
            x, y = rng.uniform(-1.5, 1.5, 2)
            z = rng.uniform(-4.0, 1.5)          # some in front of the eye, some behind it
            g.glVertex3f(float(x), float(y), float(z))
    g.glEnd()


def scene_overflows(g, W, H, seed, big=(40, 200)):
    """Overflows the clip pool, and with enough big triangles for the
    framebuffer the room for pairs too, twice."""
    rng = np.random.default_rng(seed)
    g.glMatrixMode(E["GL_PROJECTION"])
    g.glLoadIdentity()
    g.glOrtho(0.0, float(W), 0.0, float(H), 0.1, 100.0)
    g.glMatrixMode(E["GL_MODELVIEW"])
    g.glLoadIdentity()
    g.glEnable(E["GL_DEPTH_TEST"])
    g.glEnable(E["GL_BLEND"])
    g.glBlendFunc(E["GL_SRC_ALPHA"], E["GL_ONE_MINUS_SRC_ALPHA"])
    _big_triangles(g, rng, big[0], W, H)
    g.glDisable(E["GL_BLEND"])
    g.glEnable(E["GL_SCISSOR_TEST"])
    g.glScissor(W // 4, H // 4, W // 2, H // 3)
    g.glClearColor(0.3, 0.2, 0.1, 1.0)
    g.glClear(E["GL_COLOR_BUFFER_BIT"] | E["GL_DEPTH_BUFFER_BIT"])
    g.glDisable(E["GL_SCISSOR_TEST"])
    _big_triangles(g, rng, big[1], W, H)
    S._perspective(g, W, H)
    g.glDepthFunc(E["GL_LEQUAL"])
    _near_plane_fan(g, rng, 12000)               # more clipped fan triangles than the clip pool holds
    g.glRasterPos2i(0, 0)
    g.glDrawPixels(4, 4, E["GL_RGBA"], E["GL_UNSIGNED_BYTE"], g.keep(np.full(64, 200, np.uint8)))
    _big_triangles(g, rng, 10, W, H)


def _planes_and_trace(g, W, H, draw):
    ctx = g.create_context(W, H)
    try:
        g.stats_reset(ctx)
        g.glClear(E["GL_COLOR_BUFFER_BIT"] | E["GL_DEPTH_BUFFER_BIT"] | E["GL_STENCIL_BUFFER_BIT"])
        draw(g, ctx)
        planes = g.read_framebuffer(ctx, W, H)
        st = g.stats(ctx)
        how = dict(trace(g, ctx), pairs=st.bin_pairs) if g.kind == "mtgl" else None
        return planes, (st.fragments, st.triangles_raster), g.glGetError(), how
    finally:
        g.destroy_context(ctx)
        g.release()


# the second draw needs more than the first one's overflow grew the room to
BIG = (2_000, 6_000)


@pytest.mark.parametrize("seed", [1, 2])
def test_overflowed_launches_run_again_in_order(mtgl, oracle, seed):
    W, H = 320, 200
    out = [_planes_and_trace(g, W, H, lambda g, ctx: scene_overflows(g, W, H, seed, BIG)) for g in (oracle, mtgl)]
    (a, sa, ea, _), (b, sb, eb, t) = out
    assert ea == eb
    assert t["reruns"] >= 3 and t["sorted"] == 0   # the room for pairs twice, the clip pool
    d = plane_diffs(a, b)
    hist = color_histogram(a[0], b[0])
    print(f"overflows/{seed}: diffs {d} histogram {dict((i, int(v)) for i, v in enumerate(hist) if v)}", flush=True)
    assert d["depth"] == 0 and d["stencil"] == 0
    assert hist[2:].sum() == 0 and hist[1] <= max(1, a[0].size // 10000)
    assert (a[0] != a[0][0, 0]).sum() > W * H // 4   # the frame is not trivial
    assert sa == sb                                   # fragment and triangle counts equal a clean run's


@pytest.mark.parametrize("seed", [1, 2])
def test_overflowed_sorts_run_again_in_order(mtgl, oracle, seed):
    """Scattered triangles that the second frame sorts, with more pairs than a
    fresh context's sort has room for, a clear and a draw behind them."""
    W, H, n = 640, 480, 48_000

    def draw(g, ctx):
        rng = np.random.default_rng(seed)
        _ortho(g, W, H)
        for f in range(2):
            g.glClear(E["GL_COLOR_BUFFER_BIT"] | E["GL_DEPTH_BUFFER_BIT"])
            _array(g, *_triangles(rng, W, H, n, 25, False))
            g.glEnable(E["GL_SCISSOR_TEST"])
            g.glScissor(W // 3, H // 3, W // 5, H // 5)
            g.glClear(E["GL_DEPTH_BUFFER_BIT"])
            g.glDisable(E["GL_SCISSOR_TEST"])
            _array(g, *_triangles(rng, W, H, 500, 25, False))
            g.finish(ctx)

    (a, sa, ea, _), (b, sb, eb, t) = [_planes_and_trace(g, W, H, draw) for g in (oracle, mtgl)]
    assert ea == eb and sa == sb
    # the second frame's large draw at least was sorted, and its pairs are more
    # than a fresh context's sort has room for: it ran again
    assert t["sorted"] >= 2 and t["reruns"] >= 1 and t["pairs"] > 2 * 1.2 * (4 * n + 4096)
    assert plane_diffs(a, b) == {"color": 0, "depth": 0, "stencil": 0}


def test_statistics_count_each_launch_once(mtgl, oracle):
    """Fragment and pair counts after replays equal a clean run's."""
    W, H = 320, 200
    out = []
    for g in (oracle, mtgl):
        ctx = g.create_context(W, H)
        try:
            g.stats_reset(ctx)
            scene_overflows(g, W, H, 3)
            st = g.stats(ctx)
            out.append((st.fragments, st.triangles_raster))
        finally:
            g.destroy_context(ctx)
            g.release()
    print("oracle", out[0], "device", out[1])
    assert out[0] == out[1]


def test_capture_of_a_draw_that_ran_again(mtgl, oracle):
    """A differentiable capture of a draw that overflowed: the view is the one
    its second run left, not an empty one."""
    W = H = 512
    P = D.diff_params(grid=2, tex_size=16, views=1)
    P = dict(P, idx=np.ascontiguousarray(np.tile(P["idx"], 300)))   # 2,400 triangles of about 100 tiles
    tex8, _ = D.quantise(P["tex"])
    got = []
    for g in (oracle, mtgl):
        D._bind(g.lib)
        h = C.c_void_p()
        assert g.lib.mtgl_diff_create(len(P["verts"]), 16, 16, C.byref(h)) == 0
        ctx = g.create_context(W, H)
        try:
            assert g.lib.mtgl_diff_arm(g.device(ctx)) == 0
            D.draw_view(g, P, 0, W, H, tex8)
            assert g.lib.mtgl_diff_add_view(h.value, g.device(ctx)) == 0
            px = np.empty(W * H, D.GPX_DTYPE)
            assert g.lib.mtgl_diff_gbuffer(h.value, 0, px.ctypes.data) == 0
            got.append(px)
            if g is mtgl:
                assert trace(g, ctx)["reruns"] == 1
        finally:
            g.lib.mtgl_diff_destroy(h.value)
            g.destroy_context(ctx)
            g.release()
    assert (got[0]["tri"] >= 0).sum() > 10_000
    assert got[0].tobytes() == got[1].tobytes()
