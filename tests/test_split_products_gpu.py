"""float32 layers on the bf16 matrix units: every block count of a wide
network (odd ones leave half a k-step empty), its edges, and one to three
H x H layers, against the separate kernels and torch's float64 backward of
the same seeds (the bounds of test_fused_gpu._compare: network values and
losses the same in every kernel, gradients within four times the error of
torch's own float32 backward); and weights of 2^-60 to 2^20 in one layer
against float64 (beyond bf16's range: test_large_weights_gpu.py).
"""
import numpy as np
import pytest
import torch

from conftest import gpu_available

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("no HIP device", allow_module_level=True)

import problems  # noqa: E402
from test_fused_gpu import _compare, _small  # noqa: E402
from torch_de_solver_amd.nn_engine import NNEngine, mlp_arch  # noqa: E402


@pytest.mark.parametrize('width,hidden', [(33, 2), (48, 4), (49, 3), (64, 2), (65, 4), (80, 2),
                                          (81, 3), (97, 2), (112, 4), (113, 2), (128, 3),
                                          (128, 4)])
def test_wide_layers(width, hidden):
    print(f"[split products] {width} x {hidden}", flush=True)
    prob, net = _small(problems.burgers_nn, [2] + [width] * hidden + [1], seed=width + hidden,
                       nx=19, nt=13)
    _compare([prob], [net], expect='adjoint-seeds')


@pytest.mark.parametrize('width', [5, 16, 17, 32, 40, 112, 128])
def test_network_values_over_the_exponent_range(width):
    """Network values against float64 with weights of 2^-60 to 2^20 in one
    layer: relative to the sum of the output's term magnitudes, no more than
    the layer sums' float32 rounding (width * 2^-24)."""
    prob, net = _small(problems.burgers_nn, [2, width, width, 1], seed=3)
    g = torch.Generator().manual_seed(7)
    with torch.no_grad():
        scale = torch.exp2(torch.randint(-60, 1, (width, width), generator=g).float())
        net[2].weight.mul_(scale)
        net[2].weight[:, 0] *= 2.0 ** 20
    eng = NNEngine([prob], mlp_arch(net), torch.device('cuda'))
    flat = torch.cat([p.detach().reshape(-1) for p in net.parameters()]).cuda()
    u = eng.network_values(flat).cpu().double().numpy().reshape(-1)
    xs = []
    for gr in prob.groups:
        for sl, b in enumerate(gr.slot_base):
            base = np.asarray(gr.bases[b], dtype=np.float32).reshape(gr.n_entries, -1)
            xs.append(base + np.asarray(gr.slot_offset[sl], dtype=np.float64).astype(np.float32))
    x = torch.from_numpy(np.concatenate(xs, 0)).double()
    net64 = net.double()
    h = torch.tanh(net64[0](x))
    z = net64[2](h)
    ref = net64[4](torch.tanh(z)).detach().numpy().reshape(-1)
    # |du| <= |W_L| (|dz| (1 - tanh^2) + rounding of tanh and of the output sum)
    dz = width * 2.0 ** -24 * (h.abs() @ net64[2].weight.abs().t() + net64[2].bias.abs())
    slope = torch.clamp(1 - torch.tanh(z.abs() - dz.clamp(max=1.0)).clamp(min=0) ** 2, max=1.0)
    bound = ((dz * slope).clamp(max=2.0) + width * 2.0 ** -22) @ net64[4].weight.abs().t() \
        + 2.0 ** -22
    err = np.abs(u - ref) / bound.detach().numpy().reshape(-1)
    print(f"[split products] width {width}: largest error / bound {err.max():.2e}", flush=True)
    assert err.max() <= 1.0
