"""The shading's adjoint adds two neighbouring pixels' gradients pair by pair:
odd numbers of covered pixels (a last pixel without a neighbour), views with
one covered pixel or none, blocks that end inside a pair, meshes with and
without corners that follow each other in the vertex list, textures down to
one texel a side of which both taps of a row are the same.

The gradient of the images is positive, so every term added is >= 0 and a
float32 sum of n of them (any order) is within (n + 16) 2^-23 of the oracle's
sum in double, relative, the terms' own roundings (under 16) included."""
import numpy as np
import pytest

from mytinygl_amd import diff as D

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# width, height, grid, texture side, views
SIZES = [(1, 1, 4, 8, 1), (2, 1, 4, 2, 2), (9, 7, 4, 8, 1), (13, 5, 6, 4, 3), (33, 31, 16, 8, 2), (31, 65, 3, 16, 2),
         (64, 64, 48, 64, 3)]


@pytest.mark.parametrize("W,H,grid,tex,views", SIZES)
def test_gradients(mtgl, oracle, W, H, grid, tex, views):
    P = D.diff_params(grid=grid, tex_size=tex, views=views)
    P = dict(P, tex=D.quantise(P["tex"])[1])
    Vd, Vo = D.DiffViews(mtgl, P, W, H), D.DiffViews(oracle, P, W, H)
    try:
        grad = np.random.default_rng(W + H).uniform(0.5, 1.5, (views, H, W, 4)).astype(np.float32)
        leaf = [torch.from_numpy(np.ascontiguousarray(P[k], np.float32)).cuda().requires_grad_()
                for k in ("vcol", "light_rgb", "tex")]
        ref = Vo.backward_np(P["vcol"], P["light_rgb"], P["tex"], grad)
        tol = (4 * W * H * views + 16) * 2.0 ** -23
        for _ in range(2):
            for p in leaf:
                p.grad = None
            D.render(*leaf, Vd).backward(torch.from_numpy(grad).cuda())
            for name, p, r in zip(("vcol", "light_rgb", "tex"), leaf, ref):
                a = p.grad.cpu().numpy()
                assert (r >= 0).all()
                err = (np.abs(a - r) / np.maximum(r, 1e-20)).max()
                assert err <= tol, (name, err, tol)
    finally:
        Vd.close()
        Vo.close()
