"""The 'autograd' Jacobian kernel over entry counts around its workgroups'
(1 to 16 entries) and widths around its threads: the loss gradient is
J^T times each residual's weight (2 lambda / N times the residual), so
J^T w must equal the adjoint kernels' gradient; float64, 1e-11 of the
gradient's norm plus the sums' rounding (at most 5e3 terms: 5e3 eps = 1e-12);
float32 the same at 5e-5.
"""
import pytest
import torch

from conftest import gpu_available

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("no HIP device", allow_module_level=True)

from torch_de_solver_amd import workloads as W  # noqa: E402
from torch_de_solver_amd.model import Model  # noqa: E402


@pytest.mark.parametrize('dtype', ['float64', 'float32'])
@pytest.mark.parametrize('points,width', [(2, 32), (3, 7), (4, 33), (5, 32), (7, 64), (18, 65),
                                          (257, 16), (2600, 5)])
def test_gradient_is_the_jacobian_times_the_residual_weights(points, width, dtype):
    print(f"[ad jacobian] {points} points, width {width}, {dtype}", flush=True)
    d, eq, b, _, kw = W.lotka_ad(grid_res=points - 1, dtype=dtype)
    net = W.tanh_mlp([1, width, width, 2], 3,
                     torch.float64 if dtype == 'float64' else torch.float32)
    model = Model(net, d, eq, b)
    model.compile(kw['mode'], 1, kw['lambda_bound'])
    sol = model.solution_cls
    loss, _ = sol.evaluate()
    loss.backward()
    grad = torch.cat([p.grad.reshape(-1) for p in model.net.parameters()]).double()
    flat = torch.cat([p.detach().reshape(-1) for p in model.net.parameters()])
    eng = sol.engine
    jt = eng.jacobian(flat).double()
    r = eng.residuals(flat).double()
    w = torch.zeros_like(r)
    prob = sol.problem
    for gi, qi, off, cnt, col, pos in eng.tables.resid:
        q = prob.groups[gi].equations[qi]
        t = 0 if q.target is None else torch.as_tensor(q.target, device=r.device).double()
        w[off:off + cnt] = 2 * q.lam / q.denom * (r[off:off + cnt] - t)
    rel = ((jt @ w - grad).norm() / grad.norm()).item()
    print(f"  {rel:.1e}", flush=True)
    assert rel <= (1e-11 if dtype == 'float64' else 5e-5)
