"""The rounding sequence of the blend backward, bit for bit.

Gradients of scales and rotations are small differences of the blend's
per-splat sums, so single elements show any change in the order of its
roundings, however accurate; a norm over all elements does not.  One pixel
that looks along a row of splats centred on it makes every quantity of the
walk exact but the ones in question: alpha is the opacity 1/2, transmittances
are powers of two, and reciprocals of powers of two are exact.  What is left,

    S <- fma(1 - alpha, S, alpha <c, g>),   dL/dalpha = fma(-T_end <bg, g>, 1 / (1 - alpha), (<c, g> - S) T),

is restated here with one rounding each and compared with no tolerance."""
import numpy as np
import pytest
import torch

from dmgs_amd import rasterizer as RZ

pytestmark = pytest.mark.gpu

f32 = np.float32


def _fma(a, b, c):
    """a b + c rounded once: the product of two 24-bit numbers is exact in 64 bits."""
    return f32(np.float64(a) * np.float64(b) + np.float64(c))


def _walk(colors, g, bg):
    T = f32(0.5 ** len(colors))
    bg_term = f32(-T * f32(bg[0] * g[0] + bg[1] * g[1] + bg[2] * g[2]))  # exact: powers of two
    S, out = f32(0), []
    for c in colors[::-1]:
        T = f32(2 * T)
        cg = _fma(c[2], g[2], _fma(c[1], g[1], f32(c[0] * g[0])))
        out.append(_fma(bg_term, f32(2), f32(f32(cg - S) * T)))
        S = _fma(f32(0.5), S, f32(f32(0.5) * cg))
    return np.array(out[::-1], dtype=f32)


@pytest.mark.parametrize("tile_lists", [False, True])
@pytest.mark.parametrize("seed", [0, 1, 2])
def test_blend_backward_sequence(seed, tile_lists):
    print(f"case: gradient rounding seed={seed} tile_lists={tile_lists}", flush=True)
    n = 13  # transmittance 2^-13 is the last above 1e-4
    r = np.random.default_rng(seed)
    colors = r.random((n, 3), dtype=f32)
    g, bg = np.array([1.0, -0.25, 0.5], dtype=f32), np.array([1.0, 1.0, 0.5], dtype=f32)
    t = lambda a: torch.tensor(a, dtype=torch.float32, device="cuda")
    proj = torch.zeros(4, 4, device="cuda")
    proj[0, 0] = proj[1, 1] = proj[2, 2] = proj[2, 3] = 1.0  # w = z
    rs = RZ.GaussianRasterizationSettings(
        image_height=1, image_width=1, tanfovx=0.5, tanfovy=0.5, bg=t(bg), scale_modifier=1.0,
        viewmatrix=torch.eye(4, device="cuda"), projmatrix=proj, sh_degree=0, campos=torch.zeros(3, device="cuda"),
        prefiltered=False, debug=tile_lists)
    means = t([[0.0, 0.0, 1.0 + 0.1 * i] for i in range(n)])
    cov = t([[0.01, 0.0, 0.0, 0.01, 0.0, 0.01]] * n)
    opacity = torch.full((n, 1), 0.5, device="cuda", requires_grad=True)
    image, radii = RZ.GaussianRasterizer(rs)(means3D=means, means2D=torch.zeros_like(means), opacities=opacity,
                                             colors_precomp=t(colors), cov3D_precomp=cov)
    assert (radii > 0).all()
    (image * t(g).reshape(3, 1, 1)).sum().backward()
    got, want = opacity.grad.cpu().numpy().reshape(-1), _walk(colors, g, bg)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (got, want)
