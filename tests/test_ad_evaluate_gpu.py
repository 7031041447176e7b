"""Evaluate and backward in 'autograd' mode through the fused step's kernel
(its forward half for the loss, the whole of it for the gradient) against the
layer kernels, over block counts and their edges, one to four H x H layers,
entry counts around a tile and an incoming gradient other than one.  Loss
1e-6 relative, gradient 1e-5 of its norm: float32 sums of a few thousand terms
in another order, as in the fused step's own tests.
"""
import pytest
import torch

from conftest import gpu_available

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("no HIP device", allow_module_level=True)

from torch_de_solver_amd import workloads as W  # noqa: E402
from torch_de_solver_amd.model import Model  # noqa: E402


def _evaluate(monkeypatch, fused, width, hidden, n, scale):
    monkeypatch.setenv('TDX_AD_FUSED', '1' if fused else '0')
    d, eq, b, _, kw = W.poisson_ad(grid_res=n - 1)
    net = W.tanh_mlp([2] + [width] * hidden + [1], width + hidden)
    model = Model(net, d, eq, b)
    model.compile(kw['mode'], kw['lambda_operator'], kw['lambda_bound'])
    sol = model.solution_cls
    assert (sol.engine.step_kernel != 'layers') == fused
    loss, norm = sol.evaluate()
    (scale * loss).backward()
    g = torch.cat([p.grad.reshape(-1) for p in model.net.parameters()]).double()
    return loss.item(), norm.item(), g


@pytest.mark.parametrize('width,hidden,n', [(8, 1, 3), (16, 2, 4), (17, 3, 9), (48, 2, 12),
                                            (49, 5, 13), (64, 3, 25), (65, 4, 8), (100, 5, 17),
                                            (113, 2, 31), (128, 4, 20)])
def test_evaluate_matches_the_layer_kernels(width, hidden, n, monkeypatch):
    scale = 0.37
    l1, n1, g1 = _evaluate(monkeypatch, True, width, hidden, n, scale)
    l0, n0, g0 = _evaluate(monkeypatch, False, width, hidden, n, scale)
    rel = ((g1 - g0).norm() / g0.norm()).item()
    print(f"[ad evaluate] {width} x {hidden}, {n}^2: loss {abs(l1 / l0 - 1):.1e}, gradient "
          f"{rel:.1e}", flush=True)
    assert abs(l1 - l0) <= 1e-6 * abs(l0) and abs(n1 - n0) <= 1e-6 * abs(n0)
    assert rel <= 1e-5
