"""Small grids: the two-launch step (tiles with the boundary entries; Adam
with the boundary adjoint, the step's scalars and the loss) against the
separate train_step on the same plan, bit for bit, over sizes around the tile
heights the plan chooses, tiles of every requested height, both precisions
and two stencil widths; and the boundary values of chains of up to three
applications at every edge of the grid against the oracle's rolled stencils.
"""
import numpy as np
import pytest
import torch

from conftest import gpu_available

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("no HIP device", allow_module_level=True)

from oracle import tedeous_oracle as O  # noqa: E402
from torch_de_solver_amd import data as api  # noqa: E402
from torch_de_solver_amd.compiler import compile_mat  # noqa: E402
from torch_de_solver_amd.mat_engine import MatEngine  # noqa: E402

DEV = torch.device('cuda')


def _problem(n0, n1, dtype, dp, chain=(1,)):
    d = api.Domain()
    d.variable('x', [0, 1], n0 - 1, dtype=dtype)
    d.variable('t', [0, 1], n1 - 1, dtype=dtype)
    b = api.Conditions()
    b.dirichlet({'x': [0, 1], 't': 0}, value=torch.sin(np.pi * d.variable_dict['x']))
    b.dirichlet({'x': 0, 't': [0, 1]}, value=0.5)
    for name, at in (('t', 0), ('t', 1), ('x', 1)):
        bnd = {'x': [0, 1], 't': [0, 1]}
        bnd[name] = at
        b.operator(bnd, operator={'u_c': {'coeff': 1.5, 'u_c': list(chain), 'pow': 1}}, value=0.1)
    eq = api.Equation()
    eq.add({'u_tt': {'coeff': 1, 'u_tt': [1, 1], 'pow': 1},
            '-4u_xx': {'coeff': -4, 'u_xx': [0, 0], 'pow': 1},
            'u^2': {'coeff': 0.5, 'u': [None], 'pow': 2}})
    grid = d.build('mat')
    prob = compile_mat(grid, eq.equation_lst, b.build(d.variable_dict), n_eq=1,
                       derivative_points=dp, lambda_operator=1, lambda_bound=10)
    g = torch.Generator().manual_seed(n0 * 1000 + n1)
    u = torch.randn((1, n0, n1), generator=g, dtype=torch.float64)
    return d, eq, b, prob, u.to(torch.float64 if dtype == 'float64' else torch.float32)


@pytest.mark.parametrize('dtype', ['float32', 'float64'])
@pytest.mark.parametrize('size,dp,rows', [((5, 6), 2, 0), ((12, 130), 2, 0), ((57, 56), 2, 0),
                                          ((64, 113), 3, 0), ((129, 57), 2, 4),
                                          ((40, 200), 3, 8), ((300, 70), 2, 0),
                                          ((1000, 30), 2, 0), ((33, 1), 2, 0)])
def test_two_launch_step_is_the_separate_step(size, dp, rows, dtype):
    n0, n1 = size
    if n1 == 1:
        n0, n1 = 3, 900          # a grid of three rows
    print(f"[mat small] {n0}x{n1} dp {dp} rows {rows} {dtype}", flush=True)
    *_, prob, u0 = _problem(n0, n1, dtype, dp)
    eng = MatEngine(prob, DEV, tile_rows=rows)
    outs = []
    for to in (True, False):
        u = u0.to(DEV).reshape(-1).contiguous()
        m, v = torch.full_like(u, 0.01), torch.full_like(u, 0.02)
        step = torch.full((1,), 7, dtype=torch.int64, device=DEV)
        loss = torch.zeros(2, dtype=u.dtype, device=DEV)
        for _ in range(3):
            if to:
                w = torch.full_like(u, float('nan'))
                eng.train_step_to(u, w, m, v, step, 1e-3, 0.9, 0.999, 1e-8, loss)
                u = w
            else:
                eng.train_step(u, m, v, step, 1e-3, 0.9, 0.999, 1e-8, loss)
        assert int(step.item()) == 10
        outs.append([x.cpu() for x in (u, m, v, loss)])
    for a, b in zip(*outs):
        assert torch.equal(a, b), (a - b).abs().max()


@pytest.mark.parametrize('chain', [(1,), (0, 0), (0, 1, 1)])
@pytest.mark.parametrize('dp', [2, 3])
def test_boundary_chains_at_the_edges(chain, dp):
    print(f"[mat small] boundary chain {chain}, dp {dp}", flush=True)
    d, eq, b, prob, u = _problem(23, 19, 'float32', dp, chain)
    orc = O.MatOracle(dict(d.variable_dict), eq.equation_lst, [dict(c) for c in b.conditions_lst],
                      derivative_points=dp)
    *_, bv, true, keys, lens = orc.evaluate(u, 1, 10)
    eng = MatEngine(prob, DEV)
    _, _, bval = eng.fields(u.to(DEV))
    got = torch.zeros_like(bv)
    for k, (bi, col, pos) in enumerate(eng.tables.bc_entries):
        got[pos, col] = bval[k].cpu()
    np.testing.assert_array_equal(got.numpy(), bv.detach().numpy())
