"""glReadPixels and mtgl_present into pinned and ordinary memory, aligned and
not, of windows inside, across and outside the framebuffer, right after draws
that overflow the device's arrays (the read is queued behind them and must
show the frame of their second run).  Bytes before and after the window stay."""
import ctypes

import numpy as np
import pytest
import torch

from test_gpu_replay import scene_overflows
from mytinygl_amd.gl import ENUMS as E

pytestmark = pytest.mark.gpu

GUARD = 64
# (framebuffer, window x, y, width, height): every remainder of four pixels, one
# pixel, windows past each edge and outside
WINDOWS = [((97, 71), (0, 0, 97, 71)), ((64, 40), (3, 5, 33, 17)), ((64, 40), (-7, -9, 90, 66)), ((64, 40), (63, 39, 1, 1)),
           ((33, 17), (40, 2, 6, 3)), ((33, 17), (0, 20, 5, 5)), ((1, 1), (0, 0, 2, 3)), ((257, 3), (1, 0, 255, 3))]


def _draw(g, W, H):
    g.glClearColor(0.2, 0.4, 0.6, 0.8)
    g.glClear(E["GL_COLOR_BUFFER_BIT"] | E["GL_DEPTH_BUFFER_BIT"])
    scene_overflows(g, W, H, 5)


@pytest.mark.parametrize("pinned", [True, False])
@pytest.mark.parametrize("fb,win", WINDOWS)
@pytest.mark.parametrize("fmt,bpp", [("GL_RGBA", 4), ("GL_RGB", 3)])
@pytest.mark.parametrize("shift", [0, 1, 4])
def test_read_pixels(mtgl, oracle, pinned, fb, win, fmt, bpp, shift):
    n = win[2] * win[3] * bpp
    got = []
    for g in (oracle, mtgl):
        mem = torch.full((n + 2 * GUARD,), 0xA5, dtype=torch.uint8, pin_memory=pinned and g is mtgl)
        ctx = g.create_context(*fb)
        try:
            _draw(g, *fb)
            g.glReadPixels(*win, E[fmt], E["GL_UNSIGNED_BYTE"], mem.data_ptr() + GUARD + shift)
        finally:
            g.destroy_context(ctx)
            g.release()
        got.append(mem.numpy().copy())
    assert (got[0] == got[1]).all()
    assert (got[1][:GUARD + shift] == 0xA5).all() and (got[1][GUARD + shift + n:] == 0xA5).all()


@pytest.mark.parametrize("pinned", [True, False])
@pytest.mark.parametrize("fb", [(97, 71), (64, 40), (1, 1)])
@pytest.mark.parametrize("extra", [0, 4, 20])
@pytest.mark.parametrize("shift", [0, 1, 16])
def test_present(mtgl, oracle, pinned, fb, extra, shift):
    W, H = fb
    pitch = 4 * W + extra
    ctx = oracle.create_context(W, H)
    _draw(oracle, W, H)
    want = oracle.read_framebuffer(ctx, W, H)[0]
    oracle.destroy_context(ctx)
    oracle.release()
    present = mtgl.lib.mtgl_present
    present.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int32]
    mem = torch.full((H * pitch + 2 * GUARD,), 0xA5, dtype=torch.uint8, pin_memory=pinned)
    ctx = mtgl.create_context(W, H)
    try:
        _draw(mtgl, W, H)
        assert present(ctx, mem.data_ptr() + GUARD + shift, pitch) == 0
    finally:
        mtgl.destroy_context(ctx)
        mtgl.release()
    m = mem.numpy()
    rows = m[GUARD + shift:GUARD + shift + H * pitch].reshape(H, pitch)
    assert (rows[:, :4 * W] == want.view(np.uint8).reshape(H, 4 * W)).all()
    assert (rows[:, 4 * W:] == 0xA5).all() and (m[:GUARD + shift] == 0xA5).all()


def test_direct_only_within_one_allocation(mtgl):
    """Reads the device may write itself: the whole range must be one pinned
    allocation's.  A range from one into the next, with other memory between
    them, is not (the check alone: nothing is read into it)."""
    direct = mtgl.lib.mtgl_dev_host_direct
    direct.argtypes = [ctypes.c_void_p, ctypes.c_uint64]
    n = 1 << 20
    a, b = sorted((torch.empty(n, dtype=torch.uint8, pin_memory=True) for _ in range(2)), key=lambda t: t.data_ptr())
    assert b.data_ptr() - a.data_ptr() >= n
    for t in (a, b):
        assert direct(t.data_ptr(), n) == 1 and direct(t.data_ptr() + 4096, n - 4096) == 1
        assert direct(t.data_ptr() + n - 1, 1) == 1
        assert direct(t.data_ptr() + 1, n) == 0   # one byte past the allocation
    assert direct(a.data_ptr(), b.data_ptr() - a.data_ptr() + n) == 0
    assert direct(a.data_ptr() + n - 16, b.data_ptr() - a.data_ptr() - n + 32) == 0
    assert direct(torch.empty(n, dtype=torch.uint8).data_ptr(), n) == 0
