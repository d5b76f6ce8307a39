"""A draw's staged bytes (launch tables, states, client arrays) reach the device
through k_upload: 16-byte words, one or four per thread on either side of
512 KB.  Sizes at the edges of a word, of a block (256 words, 1,024 with four
per thread) and of the two forms, arrays whose start is not aligned, triangles
and points, each draw followed at once by one of other bytes."""
import numpy as np
import pytest

from conftest import plane_diffs
from mytinygl_amd.gl import ENUMS as E

pytestmark = pytest.mark.gpu

W, H = 96, 64
ALL = E["GL_COLOR_BUFFER_BIT"] | E["GL_DEPTH_BUFFER_BIT"] | E["GL_STENCIL_BUFFER_BIT"]
# 36 bytes a vertex: 14,563 of them and the tables lie about 512 KB
COUNTS = [3, 9, 27, 111, 456, 14_340, 14_562, 14_565, 14_793, 60_003]


def _arrays(rng, n, odd):
    """Interleaved position and colour (36 bytes), from an address off by odd bytes."""
    raw = np.zeros(n * 36 + 64, np.uint8)
    start = (-raw.ctypes.data) % 16 + odd
    a = raw[start:start + n * 36].view(np.float32).reshape(n, 9)
    a[:, 0] = rng.uniform(-1.1, 1.1, n)
    a[:, 1] = rng.uniform(-1.1, 1.1, n)
    a[:, 2] = rng.uniform(-1.05, 1.05, n)
    a[:, 3:7] = rng.random((n, 4))
    return raw, a


@pytest.mark.parametrize("mode", ["GL_TRIANGLES", "GL_POINTS"])
@pytest.mark.parametrize("odd", [0, 4])
@pytest.mark.parametrize("n", COUNTS)
def test_client_arrays_in_turn(mtgl, oracle, n, odd, mode):
    out = []
    for g in (oracle, mtgl):
        rng = np.random.default_rng(n + odd)
        ctx = g.create_context(W, H)
        try:
            g.glViewport(0, 0, W, H)
            g.glEnable(E["GL_DEPTH_TEST"])
            g.glEnableClientState(E["GL_VERTEX_ARRAY"])
            g.glEnableClientState(E["GL_COLOR_ARRAY"])
            g.glClear(ALL)
            for m in (n, 3 + n // 2 - (3 + n // 2) % 3, n):
                raw, a = _arrays(rng, m, odd)
                g.keep(raw)
                g.glVertexPointer(3, E["GL_FLOAT"], 36, a.ctypes.data)
                g.glColorPointer(4, E["GL_FLOAT"], 36, a.ctypes.data + 12)
                g.glDrawArrays(E[mode], 0, m)
                raw[:] = 0xFF          # (the draw has its own copy)
            out.append(g.read_framebuffer(ctx, W, H))
        finally:
            g.destroy_context(ctx)
            g.release()
    assert plane_diffs(out[0], out[1]) == {"color": 0, "depth": 0, "stencil": 0}
