"""The two ways a launch's triangles reach its tiles: k_bin, or the sort by
tile.  Which one a launch takes depends on its sizes and on how far the
triangles of a set-up block lay apart in the same draw of the frame before, so
both must leave the same pixels.  The scenes sit at the edges: one triangle and one tile,
partial squares of tiles, squares whose list is longer than a window, a
framebuffer dense enough for each square size, triangles clipped into several
records, and draws whose triangles lie together and anywhere in turn, with a
read between them (which is when the choice moves)."""
import numpy as np
import pytest

from conftest import plane_diffs, trace
from mytinygl_amd.gl import ENUMS as E
from mytinygl_amd import scenes as S

pytestmark = pytest.mark.gpu

ALL = E["GL_COLOR_BUFFER_BIT"] | E["GL_DEPTH_BUFFER_BIT"] | E["GL_STENCIL_BUFFER_BIT"]
# (framebuffer, triangles, mean size in pixels): a triangle, a square and its
# neighbours, windows of a square's list (4,096 records), squares of 4, 2 and 1
# tiles a side, scattered over many squares
SIZES = [((8, 8), 1, 6), ((33, 31), 3, 20), ((65, 129), 64, 30), ((40, 40), 65, 200), ((64, 64), 2_000, 12),
         ((32, 32), 5_000, 9), ((24, 40), 9_000, 5), ((1500, 40), 9_000, 30), ((1921, 1081), 20_000, 9),
         ((1921, 1081), 45_000, 9)]


def _ortho(g, W, H):
    g.glViewport(0, 0, W, H)
    g.glMatrixMode(E["GL_PROJECTION"])
    g.glLoadIdentity()
    g.glOrtho(0.0, float(W), 0.0, float(H), 0.1, 100.0)
    g.glMatrixMode(E["GL_MODELVIEW"])
    g.glLoadIdentity()
    g.glEnable(E["GL_DEPTH_TEST"])


def _triangles(rng, W, H, n, size, together):
    """n triangles anywhere, or in order along a path (a set-up block's lie together)."""
    if together:
        u = np.arange(n) / max(1, n - 1)
        c = np.stack([W * (0.5 + 0.45 * np.cos(7 * u)), H * (0.5 + 0.45 * np.sin(5 * u))], -1)
    else:
        c = rng.uniform(0, 1, (n, 2)) * (W, H)
    xy = c[:, None] + rng.uniform(-size, size, (n, 3, 2))
    z = -rng.uniform(0.05, 101.0, (n, 3, 1))            # some corners outside the near and far planes
    pos = np.ascontiguousarray(np.concatenate([xy, z], -1).reshape(-1, 3).astype(np.float32))
    return pos, np.ascontiguousarray(rng.random((3 * n, 4)).astype(np.float32))


@pytest.mark.parametrize("fb,n,size", SIZES)
@pytest.mark.parametrize("blend", [False, True])
def test_scattered_and_together_in_turn(mtgl, oracle, fb, n, size, blend):
    W, H = fb
    out = []
    for g in (oracle, mtgl):
        rng = np.random.default_rng(n + W)
        ctx = g.create_context(W, H)
        try:
            _ortho(g, W, H)
            if blend:
                g.glEnable(E["GL_BLEND"])
                g.glBlendFunc(E["GL_SRC_ALPHA"], E["GL_ONE_MINUS_SRC_ALPHA"])
            g.glEnableClientState(E["GL_VERTEX_ARRAY"])
            g.glEnableClientState(E["GL_COLOR_ARRAY"])
            g.glClear(ALL)
            for k, together in enumerate((False, True, True, False, False)):
                pos, col = _triangles(rng, W, H, n, size, together)
                g.glVertexPointer(3, E["GL_FLOAT"], 0, g.keep(pos))
                g.glColorPointer(4, E["GL_FLOAT"], 0, g.keep(col))
                g.glDrawArrays(E["GL_TRIANGLES"], 0, 3 * n)
                out.append(g.read_framebuffer(ctx, W, H))
                if k == 2:
                    g.glClear(ALL)
            st = g.stats(ctx)
            out.append((st.fragments, st.triangles_raster))
            if g is mtgl:
                # large draws go as the last count asks: the second (after
                # scattered triangles) and the fifth are sorted
                t = trace(g, ctx)
                assert t["binned"] + t["sorted"] == 5 + t["reruns"]
                assert t["sorted"] >= 2 and t["binned"] >= 3 if n >= 20_000 else t["sorted"] == 0
        finally:
            g.destroy_context(ctx)
            g.release()
    half = len(out) // 2
    assert out[half - 1] == out[-1]
    for a, b in zip(out[:half - 1], out[half:-1]):
        assert plane_diffs(a, b) == {"color": 0, "depth": 0, "stencil": 0}


@pytest.mark.parametrize("grid,side", [(150, 64), (290, 256)])
def test_dense_sphere(mtgl, oracle, grid, side):
    """A mesh that fills a small framebuffer (150: 45,000 triangles over 64
    tiles, squares of one tile; 290: 168,200 over 1,024, past the limit)."""
    def scene(g, W, H, seed):
        S.draw_textured_sphere(g, S.setup_textured_sphere(g, W, H, seed, grid, 64))
        if g is mtgl:
            t = trace(g, g.gl_get_current_context())
            assert (t["binned"], t["sorted"]) == ((0, 1) if grid == 290 else (1, 0))
    (a, ea), (b, eb) = S.render(oracle, scene, side, side, 3), S.render(mtgl, scene, side, side, 3)
    assert ea == eb and plane_diffs(a, b) == {"color": 0, "depth": 0, "stencil": 0}
