"""The general raster kernel's variants: scenes with no texture, with a texture,
and with per-fragment lighting, under the blend factors that have a path of
their own and others, with full and partial colour masks (which pack the
channels they keep again), and with the alpha test that makes the texture
decide depth writes.  A second frame over the first blends over bytes, not
over a clear.  Colours within one step on 0.01% of the pixels where a power is
evaluated (Phong), else equal."""
import numpy as np
import pytest

from conftest import color_histogram, plane_diffs
from mytinygl_amd.gl import ENUMS as E
from mytinygl_amd import scenes as S

pytestmark = pytest.mark.gpu

BLENDS = [("GL_SRC_ALPHA", "GL_ONE_MINUS_SRC_ALPHA"), ("GL_ONE", "GL_ONE"), ("GL_DST_COLOR", "GL_SRC_ALPHA"), None]


@pytest.mark.parametrize("need", ["plain", "texture", "phong", "phong_texture"])
@pytest.mark.parametrize("blend", BLENDS)
@pytest.mark.parametrize("mask", [(1, 1, 1, 1), (1, 0, 1, 0)])
@pytest.mark.parametrize("alpha", [False, True])
def test_variants(mtgl, oracle, need, blend, mask, alpha):
    def scene(g, W, H, seed):
        n = S.setup_textured_sphere(g, W, H, seed, 24, 32)
        g.glDisable(E["GL_FOG"])                 # (its alpha would be every fragment's)
        g.glMaterialfv(E["GL_FRONT_AND_BACK"], E["GL_DIFFUSE"], g.fv(0.9, 0.7, 0.5, 0.6))
        if "texture" not in need:
            g.glDisable(E["GL_TEXTURE_2D"])
        if "phong" in need:
            g.glShadeModel(E["GL_PHONG"])
            g.glMaterialfv(E["GL_FRONT_AND_BACK"], E["GL_SPECULAR"], g.fv(0.8, 0.6, 0.4, 1.0))
            g.glMaterialf(E["GL_FRONT_AND_BACK"], E["GL_SHININESS"], 20.5)
        if blend:
            g.glEnable(E["GL_BLEND"])
            g.glBlendFunc(E[blend[0]], E[blend[1]])
        if alpha:
            g.glEnable(E["GL_ALPHA_TEST"])
            g.glAlphaFunc(E["GL_GREATER"], 0.45)
        for k in range(2):
            g.glColorMask(*mask)
            g.glRotatef(30.0, 0.3, 1.0, 0.2)
            g.glDepthFunc(E["GL_LEQUAL" if k == 0 else "GL_ALWAYS"])
            S.draw_textured_sphere(g, n)
            g.glColorMask(1, 1, 1, 1)

    (a, ea), (b, eb) = (S.render(g, scene, 107, 61, 9, clear=(0.3, 0.7, 0.2, 0.6)) for g in (oracle, mtgl))
    assert ea == eb
    d = plane_diffs(a, b)
    hist = color_histogram(a[0], b[0])
    assert d["depth"] == 0 and d["stencil"] == 0
    assert hist[2:].sum() == 0 and hist[1] <= (max(1, a[0].size // 10000) if "phong" in need else 0)
    assert len(np.unique(a[0])) > 50
