"""Infinite weights and finite ones that bf16 rounds to infinity, in hidden
layers: the forward pass gives what float32 products give (an infinite weight
saturates its unit's tanh), at every kind of image (one block, two, odd and
even numbers of blocks)."""
import pytest
import torch

import problems
from conftest import gpu_available

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("no HIP device", allow_module_level=True)

from torch_de_solver_amd import data as api  # noqa: E402
from torch_de_solver_amd.compiler import compile_nn  # noqa: E402
from torch_de_solver_amd.nn_engine import MLPArch, NNEngine  # noqa: E402

DEV = torch.device('cuda')
MAX = torch.finfo(torch.float32).max
INF = float('inf')


def _points(g, s):
    """Inputs of the group's slot s, as the kernels form them in float32."""
    return torch.tensor(g.bases[g.slot_base[s]], dtype=torch.float32) + \
        torch.tensor(g.slot_offset[s], dtype=torch.float64).to(torch.float32)


@pytest.mark.parametrize('persistent', [0, 1])
@pytest.mark.parametrize('width', [10, 16, 31, 48, 64, 100])
def test_forward_with_infinite_and_huge_weights(width, persistent):
    d, eq, b, _ = problems.burgers_nn(api, nx=20, nt=15)
    prob = compile_nn(d.build('NN'), eq.equation_lst, b.build(d.variable_dict), 1,
                      lambda_operator=1, lambda_bound=10)
    eng = NNEngine([prob], MLPArch(d_in=2, width=width, n_out=1, n_layers=4), DEV,
                   persistent=persistent)
    net = problems.randomize_biases(problems.make_mlp([2, width, width, width, 1]))
    with torch.no_grad():
        w = net[2].weight
        w[0, 0], w[0, 1] = INF, 0.25          # a pair of neighbours in the image
        w[1, 2], w[2, 1], w[3, 3] = -INF, MAX, -0.9999 * MAX
        w[4, 4], w[4, 5] = 3.4e38, -3.4e38
        net[4].weight[5, 5] = INF
    p = torch.cat([t.detach().reshape(-1) for t in net.parameters()]).to(DEV)
    values = eng.network_values(p).cpu()
    at = 0
    for g in prob.groups:
        n = g.n_entries
        for s in range(len(g.slot_base)):
            x = _points(g, s)
            with torch.no_grad():
                ref = net(x)
            assert torch.isfinite(ref).all()
            # float32 rounding of the sums and tanh
            assert torch.allclose(values[at:at + n], ref, rtol=1e-5, atol=2e-6)
            at += n
    assert at == values.shape[0]
    loss = torch.zeros(2, device=DEV)
    eng.forward(p, loss)
    assert torch.isfinite(loss).all()
