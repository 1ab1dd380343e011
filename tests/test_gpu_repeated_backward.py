"""More than one backward through one rendered image, and a graph of the backward.

With ``retain_graph`` every backward gives the gradients of its own loss; without it a second one is an error, as for
torch's own functions.  With ``create_graph`` the gradients are those of torch's activations applied to the
rasterizer's, which are constants, whichever route renders."""
import pytest
import torch

from dmgs_amd import cameras as C
from dmgs_amd import scenes as S
from dmgs_amd.gaussian_renderer import PipelineParams, render
from helpers import grad_rel_err

pytestmark = pytest.mark.gpu


class _Plain(S.FreeGaussians):
    """A subclass: read through its getters."""


ROUTES = {"model": (S.FreeGaussians, False), "getters": (_Plain, False), "tile_lists": (_Plain, True)}


def _image(route, frozen=(), size=(140, 90)):
    cls, debug = ROUTES[route]
    m = cls(*[p.cuda() for p in S.free_scene(900, seed=4).parameters()], sh_degree=3).requires_grad_(True)
    for k in frozen:
        m.parameters()[k].requires_grad_(False)
    out = render(C.camera_at((0.4, 0.3, -3.5), *size), m, PipelineParams(debug=debug),
                 torch.tensor([0.1, 0.6, 0.3], device="cuda"))
    g = torch.randn(2, 3, size[1], size[0], generator=torch.Generator().manual_seed(1)).cuda()
    return m.parameters(), out, g


@pytest.mark.parametrize("route", ROUTES)
def test_backward_twice(route):
    print(f"case: backward twice {route}", flush=True)
    params, out, g = _image(route)
    image, points = out["render"], out["viewspace_points"]
    wanted = params + [points]
    grads = [torch.autograd.grad(image, wanted, x, retain_graph=True) for x in (g[0], g[1], g[0])]
    for a, b, c in zip(*grads):  # the order of the sums may differ from pass to pass
        assert a.any() and grad_rel_err(c, a) < 1e-6 and grad_rel_err(b, a) > 1e-2
    last = torch.autograd.grad(image, wanted, g[0] + g[1])
    for a, b, d in zip(grads[0], grads[1], last):
        assert grad_rel_err(d, a + b) < 1e-5
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(image, wanted, g[0])


@pytest.mark.parametrize("route", ["model", "getters"])
def test_graph_of_the_backward(route):
    print(f"case: create_graph {route}", flush=True)
    (params, out, g), (ref, ref_out, _) = _image(route), _image("tile_lists")
    second = []
    for ps, o in ((params, out), (ref, ref_out)):
        first = torch.autograd.grad(o["render"], ps, g[0], create_graph=True)
        second.append((first, torch.autograd.grad(sum((x ** 2).sum() for x in first), ps[3:])))
    for a, b in zip(second[0][0] + second[0][1], second[1][0] + second[1][1]):
        assert b.any() and grad_rel_err(a.detach(), b.detach()) < 1e-5


def test_graph_of_the_backward_with_frozen_tensors():
    params, out, g = _image("model", frozen=(1, 3, 4))
    asked = [params[k] for k in (0, 2, 5)]
    got = torch.autograd.grad(out["render"], asked, g[0], create_graph=True)
    for a, b in zip(got, torch.autograd.grad(out["render"], asked, g[0])):
        assert b.any() and grad_rel_err(a.detach(), b) < 1e-6
