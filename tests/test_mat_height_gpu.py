"""Tile heights of float32 'mat' plans without a generated interior: those of
the plan that rules one out (specialize = -1), whether the interior is too
small for one or the generator refuses the program.  The number of tiles
shows in the workspace (one loss pair each)."""
import pytest
import torch

import problems
from conftest import gpu_available

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("no HIP device", allow_module_level=True)

from torch_de_solver_amd import data as api  # noqa: E402
from torch_de_solver_amd import native  # noqa: E402
from torch_de_solver_amd.compiler import compile_mat  # noqa: E402
from torch_de_solver_amd.mat_engine import MatEngine  # noqa: E402

DEV = torch.device('cuda')


def _third(api, n0, n1, dp):
    """u + u_ttt: with six-point sides its reach along t is more than the
    generated kernel's strips hold."""
    d = api.Domain()
    d.variable('x', [0, 1], n0)
    d.variable('t', [0, 1], n1)
    b = api.Conditions()
    b.dirichlet({'x': [0, 1], 't': 0}, value=1)
    eq = api.Equation()
    eq.add({'u': {'coeff': 1, 'u': [None], 'pow': 1},
            'u_ttt': {'coeff': 1e-4, 'u_ttt': [1, 1, 1], 'pow': 1}})
    return d, eq, b, dp, 1


@pytest.mark.parametrize('builder,n0,n1,dp', [(problems.spec_wave, 2000, 600, 2),
                                              (problems.spec_wave, 4000, 300, 2),
                                              (_third, 1500, 1500, 6)])
def test_height_without_a_generated_interior(builder, n0, n1, dp):
    d, eq, b, dp, n_eq = builder(api, n0, n1, dp)
    prob = compile_mat(d.build('mat'), eq.equation_lst, b.build(d.variable_dict), n_eq=n_eq,
                       derivative_points=dp, lambda_operator=1, lambda_bound=10)
    auto, never = MatEngine(prob, DEV), MatEngine(prob, DEV, specialize=-1)
    assert auto.specialized_points == 0
    lib = native.lib()
    assert int(lib.tdx_mat_workspace_bytes(auto._plan)) == \
        int(lib.tdx_mat_workspace_bytes(never._plan))
    g = torch.Generator(device=DEV).manual_seed(n0)
    u = torch.randn(prob.n_eq, *[int(k) for k in prob.shape], generator=g, device=DEV)
    out = []
    for eng in (auto, never):
        loss, grad = torch.zeros(2, device=DEV), torch.empty_like(u)
        eng.forward(u, loss)
        eng.backward(u, torch.ones(1, device=DEV), grad)
        out.append((loss, grad))
    for x, y in zip(*out):
        assert torch.equal(x, y)
