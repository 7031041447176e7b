"""Which plans tdx_nn_train_step_noalloc takes: those whose workspace, with
work items of fixed size and float32 network images, is at most 64 MiB, at
every width (the images in bf16 pieces are padded to blocks of 16 units)."""
import numpy as np
import pytest
import torch

import problems
from conftest import gpu_available

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("no HIP device", allow_module_level=True)

from torch_de_solver_amd import data as api  # noqa: E402
from torch_de_solver_amd import native  # noqa: E402
from torch_de_solver_amd.compiler import compile_nn  # noqa: E402
from torch_de_solver_amd.nn_engine import MLPArch, NNEngine  # noqa: E402

DEV = torch.device('cuda')
LIMIT = 64 << 20


def _problem(nx=6, nt=5):
    d, eq, b, _ = problems.burgers_nn(api, nx=nx, nt=nt)
    return compile_nn(d.build('NN'), eq.equation_lst, b.build(d.variable_dict), 1,
                      lambda_operator=1, lambda_bound=10)


def _arch(width, hidden):
    return MLPArch(d_in=2, width=width, n_out=1, n_layers=hidden + 1)


def _instance_bytes(prob, arch):
    """Workspace of one small instance (one work item a group) with float32
    images: image, seed rows, loss pairs, gradient partials."""
    hp = (arch.width + 15) // 16 * 16
    nh = arch.n_layers - 2
    image = 2 * nh * hp * hp + hp * (1 + arch.d_in + nh + arch.n_out) + 4
    rows = sum(g.n_entries * len(g.slot_base) for g in prob.groups)
    assert all(g.n_entries <= 64 for g in prob.groups)
    return 4 * (image + rows + len(prob.groups) * (2 + arch.n_params))


def _state(eng, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    p = 0.3 * torch.randn(eng.n_inst * eng.n_params, generator=g, device=DEV)
    return [p, torch.zeros_like(p), torch.zeros_like(p),
            torch.zeros(1, dtype=torch.int64, device=DEV),
            torch.zeros(2 * eng.n_inst, device=DEV)]


def _noalloc(eng, st):
    return native.lib().tdx_nn_train_step_noalloc(
        eng._plan, *[native.ptr(t) for t in st[:4]], 1e-3, 0.9, 0.999, 1e-8, native.ptr(st[4]),
        native.stream_ptr())


@pytest.mark.parametrize('width,hidden', [(8, 3), (16, 2), (40, 4), (64, 3), (70, 3), (100, 3)])
def test_noalloc_takes_sweeps_up_to_the_limit(width, hidden):
    arch, prob = _arch(width, hidden), _problem()
    n = (LIMIT - 4096) // _instance_bytes(prob, arch)
    eng = NNEngine([prob] * n, arch, DEV)
    a, b = _state(eng), _state(eng)
    print(f"[noalloc] {n} instances of 2-{width}x{hidden}-1: workspace "
          f"{native.lib().tdx_nn_workspace_bytes(eng._plan)} bytes", flush=True)
    native.check(_noalloc(eng, a))
    eng.train_step(b[0], b[1], b[2], b[3], 1e-3, 0.9, 0.999, 1e-8, b[4])
    torch.cuda.synchronize()
    for x, y in zip(a, b):
        assert torch.equal(x, y)
    assert torch.isfinite(a[4]).all()
    del eng
    more = NNEngine([prob] * (n + max(2, n // 50)), arch, DEV)
    st = _state(more)
    assert _noalloc(more, st) == -1
    assert b'serves up to 67108864' in native.lib().tdx_last_error()
    torch.cuda.synchronize()
    assert int(st[3]) == 0
