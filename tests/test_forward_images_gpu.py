"""The separate forward kernel of wide networks: operand images in LDS (small
grids, or within 64 KB) and in global memory give the same bits, and the
persistent forward runs wherever the image fits in LDS."""
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


def _problem(dtype='float32', nx=40, nt=30):
    d, eq, b, _ = problems.burgers_nn(api, nx=nx, nt=nt, dtype=dtype)
    return compile_nn(d.build('NN'), eq.equation_lst, b.build(d.variable_dict), 1,
                      lambda_operator=1, lambda_bound=10)


def _arch(width, hidden):
    return MLPArch(d_in=2, width=width, n_out=1, n_layers=hidden + 1)


def _params(n, dtype=torch.float32):
    g = torch.Generator(device=DEV).manual_seed(n)
    return (0.3 * torch.randn(n, generator=g, device=DEV, dtype=torch.float64)).to(dtype)


@pytest.mark.parametrize('width,hidden,dtype', [(33, 2, 'float32'), (48, 4, 'float32'),
                                                (64, 3, 'float32'), (80, 3, 'float32'),
                                                (100, 2, 'float32'), (128, 2, 'float32'),
                                                (128, 3, 'float32'), (64, 3, 'float64')])
def test_images_in_lds_and_in_memory(width, hidden, dtype):
    """One instance (fewer workgroups than CUs: whatever fits is staged) and the
    same instance among 20 (more: 64 KB)."""
    prob, arch = _problem(dtype), _arch(width, hidden)
    one, many = NNEngine([prob], arch, DEV), NNEngine([prob] * 20, arch, DEV)
    p = _params(one.n_params, one.dtype)
    a, b = one.network_values(p), many.network_values(p.repeat(20))
    rows = sum(g.n_entries * len(g.slot_base) for g in prob.groups)
    assert a.shape[0] == rows and b.shape[0] == 20 * rows
    assert torch.equal(b.view(20, rows, -1), a.expand(20, -1, -1))
    assert torch.isfinite(a).all()


def _kernels(fn):
    fn()
    torch.cuda.synchronize()
    from torch.profiler import ProfilerActivity, profile
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        fn()
        torch.cuda.synchronize()
    return [e.name for e in prof.events()]


@pytest.mark.parametrize('width,hidden', [(12, 2), (32, 3), (33, 2), (48, 4), (64, 2), (64, 3),
                                          (80, 2), (100, 2), (112, 2)])
def test_persistent_forward_runs(width, hidden):
    """persistent = 1: no packing launch, the bits of persistent = -1."""
    prob, arch = _problem(), _arch(width, hidden)
    out = {}
    for ps in (-1, 1):
        eng = NNEngine([prob, prob], arch, DEV, persistent=ps)
        p = _params(2 * eng.n_params)
        loss, grad = torch.zeros(4, device=DEV), torch.empty_like(p)
        names = _kernels(lambda: eng.forward(p, loss))
        assert any('k_forward' in n for n in names)
        assert any('k_pack' in n for n in names) == (ps == -1)
        eng.backward(p, torch.ones(1, device=DEV), grad)
        out[ps] = (loss, grad)
    for x, y in zip(out[-1], out[1]):
        assert torch.equal(x, y)
