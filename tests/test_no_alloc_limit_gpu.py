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


def test_plans_keep_their_work_items_beside_the_noalloc_ones():
    """float64, 2-128x6-1: the work items that fill the device need more than
    the no-allocation array, four tiles an item do not.  A caller with a
    workspace gets the former; the no-allocation call runs the latter, the bits
    of a plan that asks for them."""
    lib = native.lib()
    d, eq, b, _ = problems.burgers_nn(api, nx=22, nt=24, dtype='float64')
    prob = compile_nn(d.build('NN'), eq.equation_lst, b.build(d.variable_dict), 1,
                      lambda_operator=1, lambda_bound=10)
    arch = _arch(128, 6)
    eng, four = NNEngine([prob], arch, DEV), NNEngine([prob], arch, DEV, chunk_tiles=4)
    cap = int(lib.tdx_noalloc_scratch_bytes())
    assert int(lib.tdx_nn_workspace_bytes(eng._plan)) > cap
    assert int(lib.tdx_nn_workspace_bytes(four._plan)) <= LIMIT
    a, b, c = ([t if t.dtype == torch.int64 else t.double() for t in _state(eng)]
               for _ in range(3))
    eng.profile(8)
    for _ in range(2):
        native.check(_noalloc(eng, a))
        four.train_step(b[0], b[1], b[2], b[3], 1e-3, 0.9, 0.999, 1e-8, b[4])
        eng.train_step(c[0], c[1], c[2], c[3], 1e-3, 0.9, 0.999, 1e-8, c[4])
    torch.cuda.synchronize()
    # launch timing counts both entry points' launches
    assert {n for _, n in eng.profile_read().values()} == {4}
    eng.profile(0)
    for x, y in zip(a, b):
        assert torch.equal(x, y)
    # the same sums in another order: each of P gradients a few 1e-15 apart,
    # Adam's first steps of 1e-3 divide by sqrt(v) + 1e-8
    assert torch.equal(a[4], c[4]) or torch.allclose(a[4], c[4], rtol=1e-9)
    assert float((a[0] - c[0]).abs().max()) <= 2 * 2 * 1e-3
    assert float(((a[1] - c[1]).norm() / c[1].norm())) <= 1e-9
