"""Backward passes whose saved tensors went through hooks: another place, another layout, another type."""
import pytest
import torch

from dmgs_amd import cameras as C
from dmgs_amd import scenes as S
from dmgs_amd.gaussian_renderer import PipelineParams, render
from helpers import grad_rel_err

pytestmark = pytest.mark.gpu


def _on_cpu():
    return torch.autograd.graph.save_on_cpu()


def _pinned():
    """Comes back contiguous, whatever its strides were."""
    return torch.autograd.graph.save_on_cpu(pin_memory=True)


def _as_double():
    """Comes back in 64 bits, where it was floating."""
    return torch.autograd.graph.saved_tensors_hooks(
        lambda t: t.clone(), lambda t: t.double() if t.dtype == torch.float32 else t)


@pytest.mark.parametrize("hooks", [_on_cpu, _pinned, _as_double])
@pytest.mark.parametrize("python_sh", [False, True])
def test_render_gradients_through_hooks(hooks, python_sh):
    print(f"case: saved-tensor hooks {hooks.__name__} python_sh={python_sh}", flush=True)
    parts = [p.cuda() for p in S.free_scene(700, seed=3, sh_degree=2).parameters()]
    cam, bg = C.camera_at((0.4, 0.3, -3.5), 73, 50), torch.tensor([0.1, 0.6, 0.3], device="cuda")
    g = torch.randn(3, 50, 73, generator=torch.Generator().manual_seed(1)).cuda()
    got = []
    for hooked in (False, True):
        m = S.FreeGaussians(*[p.clone() for p in parts], sh_degree=2).requires_grad_(True)
        pipe = PipelineParams(convert_SHs_python=python_sh)
        if hooked:
            with hooks():
                out = render(cam, m, pipe, bg)["render"]
        else:
            out = render(cam, m, pipe, bg)["render"]
        out.backward(g)
        got.append([p.grad for p in m.parameters()])
    for a, b in zip(*got):  # the same values go in: what differs is the order of the sums
        assert b.any() and grad_rel_err(a, b) < 1e-5
