"""The interpreted jet maps of the fused 'autograd' kernels take two, three or
five (point, unit) items a lane, by the network's blocks and the wavefront's
items: both sides of each boundary, evaluate and backward against the layer
kernels.  Lotka-Volterra has two jets, eight points a wavefront; Poisson five
and three.  Tolerances as in test_ad_evaluate_gpu.py: float32 sums of a few
thousand terms in another order."""
import pytest
import torch

from conftest import gpu_available

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("no HIP device", allow_module_level=True)

from torch_de_solver_amd import workloads as W  # noqa: E402
from torch_de_solver_amd.model import Model  # noqa: E402


def _evaluate(monkeypatch, fused, eq, width, hidden, n):
    monkeypatch.setenv('TDX_AD_FUSED', '1' if fused else '0')
    monkeypatch.setenv('TDX_AD_JIT', '0')
    if eq == 'lotka':
        d, e, b, _, kw = W.lotka_ad(grid_res=n - 1, dtype='float32')
        ends = (1, 2)
    else:
        d, e, b, _, kw = W.poisson_ad(grid_res=n - 1)
        ends = (2, 1)
    net = W.tanh_mlp([ends[0]] + [width] * hidden + [ends[1]], width + hidden)
    model = Model(net, d, e, b)
    model.compile(kw['mode'], kw['lambda_operator'], kw['lambda_bound'])
    sol = model.solution_cls
    assert (sol.engine.step_kernel != 'layers') == fused
    loss, norm = sol.evaluate()
    loss.backward()
    g = torch.cat([p.grad.reshape(-1) for p in model.net.parameters()]).double()
    return loss.item(), norm.item(), g


# 64 x items a lane: 128 at up to two blocks (32 units), 192 at three and four
@pytest.mark.parametrize('eq,width,hidden,n', [
    ('lotka', 15, 2, 41), ('lotka', 16, 2, 64), ('lotka', 17, 3, 41), ('lotka', 24, 2, 9),
    ('lotka', 32, 2, 100), ('lotka', 33, 2, 33), ('lotka', 64, 2, 65), ('poisson', 32, 3, 7),
    ('poisson', 33, 2, 7), ('poisson', 63, 2, 9), ('poisson', 64, 4, 6), ('poisson', 65, 2, 9)])
def test_items_a_lane(eq, width, hidden, n, monkeypatch):
    l1, n1, g1 = _evaluate(monkeypatch, True, eq, width, hidden, n)
    l0, n0, g0 = _evaluate(monkeypatch, False, eq, width, hidden, n)
    rel = ((g1 - g0).norm() / g0.norm()).item()
    print(f"[ad items] {eq} {width} x {hidden}, {n}: loss {abs(l1 / l0 - 1):.1e}, gradient "
          f"{rel:.1e}", flush=True)
    assert abs(l1 - l0) <= 1e-6 * abs(l0) and abs(n1 - n0) <= 1e-6 * abs(n0)
    assert rel <= 1e-5
