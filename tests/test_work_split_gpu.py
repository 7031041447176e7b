"""Default work items against explicit ones: a launch's split into work items
changes the order of the gradient's sums and nothing else.

The default chunk follows the problem's size (single-tile items for small
problems, whole rounds of the device for middling ones), so sizes on both
sides of a tile, of a round of work items and of the cap are taken, for the
wavefront-private, fused, block-owning and cooperative kernels.  float64
plans: the two orders differ by rounding only, 1e-11 of the gradient's norm
(sums of at most 1e5 terms of random sign, 1e5 * eps = 2e-11 at worst).
float32 plans at h = 0.1, where stencil weights stay below 100: 2e-5 (100
* eps * a few terms' cancellation), and the losses to 1e-5.
"""
import numpy as np
import pytest
import torch

from conftest import gpu_available

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("no HIP device", allow_module_level=True)

import problems  # noqa: E402
from torch_de_solver_amd import data as api  # noqa: E402
from torch_de_solver_amd.compiler import compile_nn  # noqa: E402
from torch_de_solver_amd.nn_engine import NNEngine, mlp_arch  # noqa: E402

DEV = torch.device('cuda')


def _problem(nx, nt, layers, dtype, h):
    d, eq, b, kw = problems.burgers_nn(api, nx=nx, nt=nt,
                                       dtype='float64' if dtype == torch.float64 else 'float32')
    net = problems.randomize_biases(problems.make_mlp(layers, seed=4, dtype=dtype), seed=5,
                                    scale=0.3)
    prob = compile_nn(d.build('NN'), eq.equation_lst, b.build(d.variable_dict), 1, h=h,
                      lambda_bound=10)
    return prob, net


def _run(prob, net, chunk, step):
    eng = NNEngine([prob], mlp_arch(net), DEV, chunk_tiles=chunk)
    flat = torch.cat([p.detach().reshape(-1) for p in net.parameters()]).to(DEV)
    loss = torch.zeros(2, dtype=flat.dtype, device=DEV)
    if step:
        # beta1 = 0: the first moment is the gradient
        p, m, v = flat.clone(), torch.zeros_like(flat), torch.zeros_like(flat)
        n = torch.zeros(1, dtype=torch.int64, device=DEV)
        eng.train_step(p, m, v, n, 0.0, 0.0, 0.999, 1e-8, loss)
        g = m
    else:
        eng.forward(flat, loss)
        g = torch.empty_like(flat)
        eng.backward(flat, torch.ones(1, dtype=flat.dtype, device=DEV), g)
    torch.cuda.synchronize()
    return loss.cpu().double().numpy(), g.cpu().double().numpy()


@pytest.mark.parametrize('layers', [[2, 20, 20, 1], [2, 32, 32, 32, 1], [2, 48, 48, 1],
                                    [2, 100, 100, 100, 1], [2, 24, 24, 24, 24, 24, 24, 1]])
@pytest.mark.parametrize('size', [(3, 3), (9, 17), (34, 34), (120, 61), (220, 157)])
@pytest.mark.parametrize('dtype,step', [(torch.float64, False), (torch.float32, False),
                                        (torch.float32, True)])
def test_default_split_sums_the_same_terms(layers, size, dtype, step):
    print(f"[work split] {layers} {size} {dtype} step={step}", flush=True)
    prob, net = _problem(size[0] - 1, size[1] - 1, layers, dtype, 0.1)
    l0, g0 = _run(prob, net, 0, step)
    l1, g1 = _run(prob, net, 7, step)
    rel = np.linalg.norm(g0 - g1) / np.linalg.norm(g1)
    print(f"  gradient {rel:.1e}, loss {np.abs(l0 / l1 - 1).max():.1e}", flush=True)
    tol = 1e-11 if dtype == torch.float64 else 2e-5
    assert rel <= tol
    np.testing.assert_allclose(l0, l1, rtol=1e-12 if dtype == torch.float64 else 1e-5)
