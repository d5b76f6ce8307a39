"""How launches are sized: grids by what a draw can cover, whatever its number
of triangles."""
import ctypes

import pytest

from mytinygl_amd.gl import ENUMS as E

pytestmark = pytest.mark.gpu

ALL = E["GL_COLOR_BUFFER_BIT"] | E["GL_DEPTH_BUFFER_BIT"] | E["GL_STENCIL_BUFFER_BIT"]


def trace(g, ctx):
    fn = g.lib.mtgl_dev_launch_trace
    fn.argtypes = [ctypes.c_void_p, ctypes.POINTER(ctypes.c_uint64)]
    out = ctypes.c_uint64()
    assert fn(g.device(ctx), ctypes.byref(out)) == 0
    return out.value


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
        assert trace(mtgl, ctx) >= min(1024, max(1, tiles if tiles < 64 else tiles & ~63))
    finally:
        mtgl.destroy_context(ctx)
        mtgl.release()
