"""Two losses evaluated before their backwards ('autograd' mode): the gradients
are those of the losses alone, and the fused kernel, which forms its own jets,
runs no forward pass again (the layer kernels do)."""
import pytest
import torch

from conftest import gpu_available

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("no HIP device", allow_module_level=True)

from torch_de_solver_amd import workloads as W  # noqa: E402
from torch_de_solver_amd.model import Model  # noqa: E402


@pytest.mark.parametrize('fused', [True, False])
def test_two_losses_before_the_backwards(fused, monkeypatch):
    monkeypatch.setenv('TDX_AD_FUSED', '1' if fused else '0')
    d, eq, b, _, kw = W.poisson_ad(grid_res=11)
    model = Model(W.tanh_mlp([2, 32, 32, 1], 3), d, eq, b)
    model.compile(kw['mode'], kw['lambda_operator'], kw['lambda_bound'])
    eng = model.solution_cls.engine
    assert (eng.step_kernel != 'layers') == fused
    a = torch.cat([p.detach().reshape(-1) for p in model.net.parameters()])
    points = [a, 1.25 * a]
    alone = []
    for q in points:
        q = q.clone().requires_grad_()
        eng.loss(q)[0, 0].backward()
        alone.append(q.grad)
    passes = []
    forward = eng.forward
    monkeypatch.setattr(eng, 'forward', lambda *args: (passes.append(1), forward(*args)))
    leaves = [q.clone().requires_grad_() for q in points]
    losses = [eng.loss(q)[0, 0] for q in leaves]
    for loss in losses:
        loss.backward()
    for q, g in zip(leaves, alone):
        assert torch.equal(q.grad, g)
    assert len(passes) == (2 if fused else 4)
