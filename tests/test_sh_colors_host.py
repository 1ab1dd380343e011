"""The Python SH colours' second-order path, which is torch operations, on the CPU."""
from types import SimpleNamespace

import pytest
import torch

from dmgs_amd import gaussian_renderer as GR


@pytest.mark.parametrize("degree", [0, 2])
@pytest.mark.parametrize("needs", [(True, True), (True, False), (False, True)])
def test_create_graph_with_a_frozen_input(needs, degree):
    g = torch.Generator().manual_seed(degree)
    feats = torch.randn(5, 3, 9, generator=g, dtype=torch.float64).requires_grad_(needs[0])
    xyz = torch.randn(5, 3, generator=g, dtype=torch.float64).requires_grad_(needs[1])
    campos = torch.tensor([0.1, 3.0, -0.4], dtype=torch.float64)
    grad = torch.randn(5, 3, generator=g, dtype=torch.float64)
    ctx = SimpleNamespace(saved_tensors=(feats, xyz, campos, None), degree=degree,
                          needs_input_grad=needs + (False, False))
    got = GR._ShSigmoid.backward(ctx, grad)
    assert got[2:] == (None, None)
    colors = GR._torch_colors(feats, xyz, campos, degree)
    for x, need, y in zip((feats, xyz), needs, got):
        if not need or (x is xyz and degree == 0):  # constant colours have no gradient in the position
            assert y is None
            continue
        want, = torch.autograd.grad(colors, x, grad, create_graph=True)
        assert torch.equal(y, want)
        assert torch.equal(*(torch.autograd.grad((z ** 2).sum(), x, retain_graph=True)[0] for z in (y, want)))
