"""What a user of this framework has it do, as cases that can be timed.

Every case is one problem (its equation, grid, network and precision) and one
call on it, through the entry points a program uses:

* ``train``: a short ``Model.train`` with Adam, as a script calls it (initial
  loss, captured step, replays), each pass from the problem's first weights:
  small problems, where launches count.
* ``step``: one fused training step of the compiled problem
  (``engine.train_step``, ``train_step_to`` on a grid, ``SweepSolver.step``
  for a sweep): loss, new weights and both Adam moments.
* ``grad``: ``Solution.evaluate`` and ``backward``, the pass under any other
  optimizer or callback (L-BFGS, schedulers, adaptive lambdas): loss and
  gradients.
* ``jacobian``: the residual Jacobian of a natural-gradient step.

Problems: Legendre, Burgers and Korteweg-de Vries on shifted-network stencils
('NN'), the wave equation on a grid tensor ('mat'), Poisson and Lotka-Volterra
by differentiation of the network ('autograd'), and a sweep of independent
Burgers solves of uneven sizes.  ``exact`` computes the same in 64 bits with
plain torch; the points and their shifted copies are inputs there and stay in
the problem's precision.
"""

import math

import numpy as np
import torch

from torch_de_solver_amd import workloads
from torch_de_solver_amd.data import Conditions, Domain, Equation
from torch_de_solver_amd.model import Model
from torch_de_solver_amd.optimizers import Optimizer
from torch_de_solver_amd.sweep import SweepSolver

LR, BETA1, BETA2, EPS = 1e-3, 0.9, 0.999, 1e-8
DONE = 100          # steps behind the Adam state of a 'step' case


def listed():
    return [
        # the smallest solve: an ordinary differential equation on 100 points,
        # trained by Model.train; launches and latency
        dict(name='legendre_train', call='train', eq='legendre', n0=100, n1=1, width=100,
             hidden=2, dtype='float32', epochs=51),
        # a small grid tensor under Model.train, one step a few microseconds
        # of work
        dict(name='wave_train', call='train', eq='wave', n0=128, n1=128, dtype='float32',
             epochs=301),
        # a large grid tensor: the streaming case
        dict(name='wave_large_step', call='step', eq='wave', n0=8192, n1=8192, dtype='float32'),
        # a ragged grid in double precision under a torch optimizer
        dict(name='wave_f64_grad', call='grad', eq='wave', n0=777, n1=1001, dtype='float64'),
        # the parameter sweep: 256 small networks, uneven grids, one plan
        dict(name='sweep_step', call='step', eq='sweep', count=256, mix=0, width=32, hidden=3,
             dtype='float32'),
        # a few instances only: the grid does not fill the device as it likes
        dict(name='sweep_small_step', call='step', eq='sweep', count=9, mix=5, width=32,
             hidden=3, dtype='float32'),
        # single solves with the wide networks of the usual scripts
        dict(name='burgers_step', call='step', eq='burgers', n0=256, n1=100, width=100, hidden=4,
             dtype='float32'),
        dict(name='kdv_step', call='step', eq='kdv', n0=512, n1=128, width=64, hidden=4,
             dtype='float32'),
        # evaluate and backward for a torch optimizer, odd grid, narrow network
        dict(name='burgers_grad', call='grad', eq='burgers', n0=201, n1=77, width=32, hidden=3,
             dtype='float32'),
        # differentiation of the network itself: fused step, and evaluate and
        # backward
        dict(name='poisson_step', call='step', eq='poisson', n0=201, n1=201, width=100, hidden=5,
             dtype='float32'),
        dict(name='poisson_grad', call='grad', eq='poisson', n0=133, n1=91, width=64, hidden=3,
             dtype='float32'),
        # the Jacobian of a natural-gradient step on a system of two equations
        dict(name='lotka_jacobian', call='jacobian', eq='lotka', n0=501, n1=1, width=32,
             hidden=2, dtype='float32'),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(['train', 'wave', 'sweep', 'nn', 'nn', 'nn', 'poisson', 'poisson',
                       'lotka'])
    if kind == 'train':
        if rng.random() < 0.5:
            return dict(call='train', eq='legendre', n0=size(40, 400), n1=1,
                        width=rng.choice([16, 32, 50, 64, 100]), hidden=rng.randint(2, 4),
                        dtype='float32', epochs=51)
        return dict(call='train', eq='wave', n0=size(32, 300), n1=size(32, 300),
                    dtype='float32', epochs=201)
    if kind == 'wave':
        if rng.random() < 0.6:
            return dict(call='step', eq='wave', n0=size(300, 8000), n1=size(300, 8000),
                        dtype='float32')
        return dict(call='grad', eq='wave', n0=size(100, 2000), n1=size(100, 2000),
                    dtype=rng.choice(['float32', 'float64']))
    if kind == 'sweep':
        return dict(call='step', eq='sweep', count=size(2, 200), mix=rng.randint(1, 1 << 20),
                    width=rng.choice([20, 32, 32]), hidden=rng.randint(2, 3), dtype='float32')
    if kind == 'nn':
        eq = rng.choice(['burgers', 'burgers', 'kdv'])
        f64 = eq == 'burgers' and rng.random() < 0.15
        # (third differences over h^3 leave a 32-bit KdV operator loss, apart
        # from the conditions', only a digit or two: fused steps only)
        return dict(call='grad' if f64 else 'step' if eq == 'kdv' else
                    rng.choice(['step', 'grad']), eq=eq,
                    n0=size(40, 256), n1=size(20, 128),
                    width=64 if eq == 'kdv' else rng.choice([20, 32, 48, 64, 100, 128]),
                    hidden=4 if eq == 'kdv' else rng.randint(2, 4),
                    dtype='float64' if f64 else 'float32')
    if kind == 'poisson':
        return dict(call=rng.choice(['step', 'grad']), eq='poisson', n0=size(30, 201),
                    n1=size(30, 201), width=rng.choice([32, 64, 100, 128]),
                    hidden=rng.randint(2, 5), dtype='float32')
    return dict(call='jacobian', eq='lotka', n0=size(60, 501), n1=1, width=rng.choice([16, 32]),
                hidden=2, dtype=rng.choice(['float32', 'float64']))


# ---------------------------------------------------------------------------
# the problems, as a script sets them up
# ---------------------------------------------------------------------------

def _layers(case):
    ends = {'legendre': (1, 1), 'lotka': (1, 2)}.get(case['eq'], (2, 1))
    return [ends[0]] + [case['width']] * case['hidden'] + [ends[1]]


def _dtype(case):
    return torch.float64 if case['dtype'] == 'float64' else torch.float32


def _wave(case):
    d, eq, b = Domain(), Equation(), Conditions()
    d.variable('x', [0, 1], case['n0'] - 1, dtype=case['dtype'])
    d.variable('t', [0, 1], case['n1'] - 1, dtype=case['dtype'])
    b.dirichlet({'x': [0, 1], 't': 0}, value=torch.sin(np.pi * d.variable_dict['x']))
    b.dirichlet({'x': 0, 't': [0, 1]}, value=0)
    b.dirichlet({'x': 1, 't': [0, 1]}, value=0)
    b.operator({'x': [0, 1], 't': 0}, operator={'u_t': {'coeff': 1, 'u_t': [1], 'pow': 1}},
               value=0)
    eq.add({'u_tt': {'coeff': 1, 'u_tt': [1, 1], 'pow': 1},
            '-4u_xx': {'coeff': -4, 'u_xx': [0, 0], 'pow': 1}})
    return d, eq, b, None, dict(mode='mat', lambda_operator=1, lambda_bound=100)


def _poisson(case):
    d, eq, b = Domain(), Equation(), Conditions()
    d.variable('x', [0, 1], case['n0'] - 1)
    d.variable('y', [0, 1], case['n1'] - 1)
    for side in ({'x': 0, 'y': [0, 1]}, {'x': 1, 'y': [0, 1]}, {'x': [0, 1], 'y': 0},
                 {'x': [0, 1], 'y': 1}):
        b.dirichlet(side, value=0)
    eq.add({'-u_xx': {'coeff': -1., 'u_xx': [0, 0], 'pow': 1, 'var': 0},
            '-u_yy': {'coeff': -1., 'u_yy': [1, 1], 'pow': 1, 'var': 0},
            '-f': {'coeff': lambda g: -2 * np.pi ** 2 * torch.sin(np.pi * g[:, 0]) *
                   torch.sin(np.pi * g[:, 1]), 'u': [None], 'pow': 0, 'var': 0}})
    return d, eq, b, None, dict(mode='autograd', lambda_operator=1, lambda_bound=100)


def _network(layers, seed, dtype):
    """Linear/Tanh stack as the scripts make it: Xavier-normal weights, small
    biases as after some training."""
    g = torch.Generator().manual_seed(seed)
    mods = []
    for i, (a, b) in enumerate(zip(layers[:-1], layers[1:])):
        lin = torch.nn.Linear(a, b)
        with torch.no_grad():
            lin.weight.copy_(torch.randn(b, a, generator=g) * math.sqrt(2.0 / (a + b)))
            lin.bias.copy_(0.1 * torch.randn(b, generator=g))
        mods.append(lin)
        if i < len(layers) - 2:
            mods.append(torch.nn.Tanh())
    return torch.nn.Sequential(*mods).to(dtype)


def _grid_values(case, seed):
    """Start of a grid solve: the initial profile along x, decaying in t, with
    seeded noise."""
    g = torch.Generator().manual_seed(seed)
    n0, n1 = case['n0'], case['n1']
    x = torch.sin(np.pi * torch.linspace(0, 1, n0)).reshape(n0, 1)
    t = torch.cos(2 * np.pi * torch.linspace(0, 1, n1)).reshape(1, n1)
    u = x * t * (0.5 + 0.5 * torch.rand((), generator=g))
    noise = torch.Generator(device='cuda').manual_seed(seed)
    u = u.cuda() + 0.01 * torch.randn(n0, n1, generator=noise, device='cuda')
    return u.reshape(1, n0, n1).to(_dtype(case))


def _problem(case, seed):
    eq = case['eq']
    if eq == 'legendre':
        d, e, b, _, kw = workloads.legendre(n_points=case['n0'] - 1)
    elif eq == 'burgers':
        d, e, b, _, kw = workloads.burgers(nx=case['n0'], nt=case['n1'], layers=(2, 8, 1),
                                           dtype=case['dtype'])
    elif eq == 'kdv':
        d, e, b, _, kw = workloads.kdv(nx=case['n0'], nt=case['n1'], dtype=case['dtype'])
    elif eq == 'lotka':
        d, e, b, _, kw = workloads.lotka_ad(grid_res=case['n0'] - 1, dtype=case['dtype'])
    elif eq == 'poisson':
        d, e, b, _, kw = _poisson(case)
    else:
        d, e, b, _, kw = _wave(case)
    net = _grid_values(case, seed) if eq == 'wave' else _network(_layers(case), seed, _dtype(case))
    return d, e, b, net, kw


def _sweep_sizes(case):
    return workloads.sweep_instances(case['count'], case['mix'])


def _moments(count, seed, dtype, device='cuda'):
    """Adam's moments in the middle of a training run."""
    g = torch.Generator(device=device).manual_seed(seed + 17)
    m = 0.1 * torch.randn(count, generator=g, device=device)
    v = 0.01 * (0.5 + torch.rand(count, generator=g, device=device))
    return m.to(dtype), v.to(dtype)


def prepare(case, seed):
    dtype = _dtype(case)
    if case['eq'] == 'sweep':
        problems = []
        for k, s in enumerate(_sweep_sizes(case)):
            d, e, b, _, kw = workloads.burgers(nx=s.nx, nt=s.nt, nu=s.nu, layers=(2, 8, 1))
            problems.append((d, e, b, _network(_layers(case), 1000 * seed + k, dtype), kw))
        solver = SweepSolver(problems)
        m, v = _moments(solver.params.numel(), seed, dtype)
        solver.exp_avg.copy_(m)
        solver.exp_avg_sq.copy_(v)
        solver.step_count.fill_(DONE)
        return dict(case=case, solver=solver)
    d, e, b, net, kw = _problem(case, seed)
    model = Model(net, d, e, b)
    model.verbose = False
    model.compile(kw.pop('mode'), **kw)
    state = dict(case=case, model=model, sol=model.solution_cls, eng=model.solution_cls.engine)
    if case['call'] == 'train':
        state['optimizer'] = Optimizer('Adam', {'lr': LR})
        leaves = [model.net] if case['eq'] == 'wave' else list(model.net.parameters())
        state['first'] = [(p, p.detach().clone()) for p in leaves]
    elif case['call'] == 'step':
        flat = model.net if case['eq'] == 'wave' else \
            torch.cat([p.detach().reshape(-1) for p in model.net.parameters()])
        m, v = _moments(flat.numel(), seed, dtype)
        state.update(params=flat.contiguous(), m=m.view_as(flat), v=v.view_as(flat),
                     steps=torch.full((1,), DONE, dtype=torch.int64, device='cuda'),
                     loss=torch.zeros(2, dtype=dtype, device='cuda'))
        if case['eq'] == 'wave':
            state['other'] = torch.empty_like(flat)
    elif case['call'] == 'jacobian':
        state['params'] = torch.cat([p.detach().reshape(-1) for p in model.net.parameters()])
    elif case['eq'] == 'wave':
        model.net.requires_grad_()
    return state


def run(state):
    case = state['case']
    if case['call'] == 'train':
        model = state['model']
        for p, first in state['first']:
            p.data.copy_(first)
        model.train(state['optimizer'], case['epochs'])
        if case['eq'] == 'wave':
            return [model.cur_loss, model.net]
        return [model.cur_loss] + [p.detach() for p in model.net.parameters()]
    if case['call'] == 'grad':
        sol, net = state['sol'], state['model'].net
        leaves = [net] if case['eq'] == 'wave' else list(net.parameters())
        for p in leaves:
            p.grad = None
        loss, norm = sol.evaluate()
        loss.backward()
        return [loss.detach(), norm] + [p.grad for p in leaves]
    if case['call'] == 'jacobian':
        return [state['eng'].jacobian(state['params'])]
    if case['eq'] == 'sweep':
        s = state['solver']
        s.step(lr=LR, betas=(BETA1, BETA2), eps=EPS)
        return [s.loss_buf, s.params, s.exp_avg, s.exp_avg_sq]
    s = state
    if case['eq'] == 'wave':
        s['eng'].train_step_to(s['params'], s['other'], s['m'], s['v'], s['steps'], LR, BETA1,
                               BETA2, EPS, s['loss'])
        s['params'], s['other'] = s['other'], s['params']
    else:
        s['eng'].train_step(s['params'], s['m'], s['v'], s['steps'], LR, BETA1, BETA2, EPS,
                            s['loss'])
    return [s['loss'], s['params'], s['m'], s['v']]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _rows(case):
    """(points of the operator, network evaluations or jets per point, points
    of the conditions)."""
    n0, n1 = case['n0'], case['n1']
    return {'legendre': (n0, 5, 2),                       # u, x+-h, x+-2h
            'burgers': ((n0 - 2) * (n1 - 2), 7, n0 + 2 * n1),
            'kdv': ((n0 - 2) * (n1 - 2), 7, n0 + 2 * n1),
            'poisson': (n0 * n1, 5, 2 * (n0 + n1)),
            'lotka': (n0, 2, 2)}[case['eq']]


def _net_work(layers, rows):
    """Forward, transposed and weight products of a step, per row of inputs."""
    return 3.0 * rows * sum(2 * a * b for a, b in zip(layers[:-1], layers[1:]))


def work(case):
    size = 8 if case['dtype'] == 'float64' else 4
    if case['eq'] == 'wave':
        n = case['n0'] * case['n1']
        per = {'step': 6, 'train': 6, 'grad': 2}[case['call']]
        times = case['epochs'] - 1 if case['call'] == 'train' else 1
        return {'bytes': times * per * size * n, 'flops': times * 40.0 * n}
    layers = _layers(case)
    count = sum(a * b + b for a, b in zip(layers[:-1], layers[1:]))
    if case['eq'] == 'sweep':
        parts = [_rows(dict(eq='burgers', n0=s.nx, n1=s.nt)) for s in _sweep_sizes(case)]
        flops = sum(_net_work(layers, p * k + c) for p, k, c in parts)
        values = sum(2 * (p + c) for p, k, c in parts) + 6 * count * len(parts)
        return {'bytes': size * values, 'flops': flops}
    points, per, bnd = _rows(case)
    rows = points * per + bnd
    if case['call'] == 'jacobian':
        # forward and transposed products of each residual, and its row of J
        resid = 2 * points + bnd
        return {'bytes': size * resid * count, 'flops': _net_work(layers, resid * 2) }
    if case['eq'] == 'poisson':
        rows = (points + bnd) * per
    times = case['epochs'] - 1 if case['call'] == 'train' else 1
    values = 2 * (points + bnd) + (2 if case['call'] == 'grad' else 6) * count
    return {'bytes': times * size * values, 'flops': times * _net_work(layers, rows)}


def tolerance(case):
    """About four times the largest error against 64 bits seen over the ranges
    of ``draw``.  The network problems take differences of 32-bit network
    values over h (1e-3; KdV: over h^3, 1e-6), which is what remains of them
    in gradients.  Of Legendre runs of 50 steps the same is said from one
    order of the gradient's sums to another (work items of one tile and of
    eight; after 150 steps losses are up to 5.6e-2 apart, single weights 9e-2)."""
    eq, wide = case['eq'], case['dtype'] == 'float64'
    if case['call'] == 'train':
        return {'rel': 0.016, 'max': 0.05} if eq == 'legendre' else {'rel': 2e-3}
    if eq == 'wave':
        return {'rel': 4e-15} if wide else {'rel': 1.2e-6, 'max': 2e-3}
    if eq in ('poisson', 'lotka'):
        return {'rel': 2e-15 if wide else 2e-6}
    if wide:
        return {'rel': 4e-12}
    if eq == 'kdv':
        return {'rel': 5e-3}
    return {'rel': 2e-3 if case['call'] == 'grad' else 5e-5}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

def _net64(params, x):
    n = len(params) // 2
    for i in range(n):
        x = x @ params[2 * i].t() + params[2 * i + 1]
        if i < n - 1:
            x = torch.tanh(x)
    return x


def _axis(lo, hi, n, dtype):
    return torch.linspace(lo, hi, n, dtype=dtype)


def _shifted(pts, axis, k, h):
    """Points moved by k steps along an axis, in the points' own precision."""
    out = pts.clone()
    out[:, axis] = pts[:, axis] + k * h
    return out


def _stencil_loss(case, params, nu=0.01 / math.pi):
    """(loss, normalized loss) of the 'NN' problems: central differences of the
    network at shifted points, squared residual means and condition means."""
    dt, eq = _dtype(case), case['eq']
    u = lambda p: _net64(params, p.cuda().double())[:, 0]  # noqa: E731
    if eq == 'legendre':
        h, lam = 1e-3, 10.0
        pts = _axis(-1, 1, case['n0'], dt).reshape(-1, 1)
        x = pts[:, 0].cuda().double()
        at = {k: u(_shifted(pts, 0, k, h)) for k in (-2, -1, 0, 1, 2)}
        u1 = (at[1] - at[-1]) / (2 * h)
        u2 = (at[2] - 2 * at[0] + at[-2]) / (4 * h * h)
        op = (1 - x * x) * u2 - 2 * x * u1 + 12 * at[0]
        ends = u(torch.tensor([[-1.0], [1.0]], dtype=dt)) - torch.tensor([-1.0, 1.0]).cuda()
        cond = [(ends, 2)]
    else:
        n0, n1 = case['n0'], case['n1']
        t = _axis(0, 1, n1, dt)
        x = (20.0 * torch.arange(n0, dtype=torch.float32) / n0).to(dt) if eq == 'kdv' \
            else _axis(-1, 1, n0, dt)
        h, lam = (0.01, 100.0) if eq == 'kdv' else (1e-3, 10.0)
        pts = torch.cartesian_prod(x[1:-1], t[1:-1])
        u0 = u(pts)
        ut = (u(_shifted(pts, 1, 1, h)) - u(_shifted(pts, 1, -1, h))) / (2 * h)
        p1, m1 = u(_shifted(pts, 0, 1, h)), u(_shifted(pts, 0, -1, h))
        ux = (p1 - m1) / (2 * h)
        start = torch.stack([x, torch.zeros_like(x)], 1)
        if eq == 'kdv':
            p3, m3 = u(_shifted(pts, 0, 3, h)), u(_shifted(pts, 0, -3, h))
            op = ut + 6 * u0 * ux + (p3 - 3 * p1 + 3 * m1 - m3) / (8 * h ** 3)
            side = lambda c: u(torch.stack([torch.full_like(t, c), t], 1))  # noqa: E731
            first = u(start) - (0.5 / torch.cosh(0.5 * (x - 10.0)) ** 2).cuda().double()
            most = max(n0, n1)
            cond = [(side(0.0) - side(20.0), most), (first, most)]
        else:
            p2, m2 = u(_shifted(pts, 0, 2, h)), u(_shifted(pts, 0, -2, h))
            op = ut + u0 * ux - nu * (p2 - 2 * u0 + m2) / (4 * h * h)
            side = lambda c: u(torch.stack([torch.full_like(t, c), t], 1))  # noqa: E731
            first = u(start) + torch.sin(np.pi * x).cuda().double()
            cond = [(torch.cat([first, side(-1.0), side(1.0)]), n0 + 2 * n1)]
    main = (op * op).mean()
    rest = sum((c * c).sum() / n for c, n in cond)
    return main + lam * rest, main + rest


def _poisson_loss(case, params):
    n0, n1 = case['n0'], case['n1']
    x, y = _axis(0, 1, n0, torch.float32), _axis(0, 1, n1, torch.float32)
    pts = torch.cartesian_prod(x, y).cuda().double().requires_grad_()
    u = _net64(params, pts)
    g = torch.autograd.grad(u.sum(), pts, create_graph=True)[0]
    uxx = torch.autograd.grad(g[:, 0].sum(), pts, create_graph=True)[0][:, 0]
    uyy = torch.autograd.grad(g[:, 1].sum(), pts, create_graph=True)[0][:, 1]
    f = 2 * np.pi ** 2 * torch.sin(np.pi * pts[:, 0]) * torch.sin(np.pi * pts[:, 1])
    op = -uxx - uyy - f.detach()
    z = torch.zeros
    sides = torch.cat([torch.stack([z(n1), y], 1), torch.stack([z(n1) + 1, y], 1),
                       torch.stack([x, z(n0)], 1), torch.stack([x, z(n0) + 1], 1)])
    b = _net64(params, sides.cuda().double())[:, 0]
    main, rest = (op * op).mean(), (b * b).mean()
    return main + 100.0 * rest, main + rest


def _wave_loss(case, u):
    """Differences of the grid tensor, one-sided at its ends, applied twice."""
    def diff(v, axis, h):
        inner = (v.narrow(axis, 2, v.shape[axis] - 2) - v.narrow(axis, 0, v.shape[axis] - 2))
        lo = (v.narrow(axis, 1, 1) - v.narrow(axis, 0, 1)) / h
        n = v.shape[axis]
        hi = (v.narrow(axis, n - 1, 1) - v.narrow(axis, n - 2, 1)) / h
        return torch.cat([lo, inner / (2 * h), hi], axis)

    dt, n0, n1 = _dtype(case), case['n0'], case['n1']
    x, t = _axis(0, 1, n0, dt), _axis(0, 1, n1, dt)
    h0, h1 = (float(a.float()[1] - a.float()[0]) for a in (x, t))   # a 32-bit step, by definition
    w = u[0]
    ut = diff(w, 1, h1)
    op = diff(ut, 1, h1) - 4 * diff(diff(w, 0, h0), 0, h0)
    main = (op * op).mean()
    values = torch.cat([w[:, 0] - torch.sin(np.pi * x).cuda().double(), w[0], w[-1]])
    most = n0 + 2 * n1
    rest = (values * values).sum() / most + (ut[:, 0] ** 2).sum() / most
    return main + 100.0 * rest, main + rest


def _adam(p, g, m, v, step):
    m = BETA1 * m + (1 - BETA1) * g
    v = BETA2 * v + (1 - BETA2) * g * g
    den = (v / (1 - BETA2 ** step)).sqrt() + EPS
    return p - LR * (m / (1 - BETA1 ** step)) / den, m, v


def _weights64(case, seed):
    net = _network(_layers(case), seed, _dtype(case))
    return [p.detach().cuda().double().requires_grad_() for p in net.parameters()]


def _flat(tensors):
    return torch.cat([t.reshape(-1) for t in tensors])


def _lotka_jacobian(case, params):
    """Rows of d residual / d weights, transposed: both equations at every
    point, then the two conditions."""
    t = _axis(0, 1, case['n0'], _dtype(case)).reshape(-1, 1).cuda().double().requires_grad_()
    u = _net64(params, t)
    x, y = u[:, 0], u[:, 1]
    dx = torch.autograd.grad(x.sum(), t, create_graph=True)[0][:, 0]
    dy = torch.autograd.grad(y.sum(), t, create_graph=True)[0][:, 0]
    start = _net64(params, torch.zeros(1, 1, dtype=torch.float64, device='cuda'))[0]
    resid = torch.cat([dx - 20 * x + 20 * x * y, dy + 20 * y - 20 * x * y, start])
    rows = [_flat(torch.autograd.grad(r, params, retain_graph=True, allow_unused=True,
                                      materialize_grads=True)) for r in resid]
    return torch.stack(rows, 1)


def exact(case, seed):
    if case['eq'] == 'sweep':
        losses, done = [], []
        layers = _layers(case)
        count = sum(a * b + b for a, b in zip(layers[:-1], layers[1:]))
        m, v = _moments(count * case['count'], seed, torch.float32)
        for k, s in enumerate(_sweep_sizes(case)):
            p = _weights64(case, 1000 * seed + k)
            one = dict(eq='burgers', n0=s.nx, n1=s.nt, dtype=case['dtype'])
            loss, norm = _stencil_loss(one, p, s.nu)
            g = _flat(torch.autograd.grad(loss, p))
            at = slice(k * count, (k + 1) * count)
            done.append(_adam(_flat(p).detach(), g, m[at].double(), v[at].double(), DONE + 1))
            losses += [loss.detach(), norm.detach()]
        return [torch.stack(losses)] + [torch.cat(c) for c in zip(*done)]
    wave = case['eq'] == 'wave'
    if wave:
        p = [_grid_values(case, seed).double().requires_grad_()]
        pair = lambda q: _wave_loss(case, q[0])  # noqa: E731
    else:
        p = _weights64(case, seed)
        if case['eq'] == 'lotka':
            return [_lotka_jacobian(case, p)]
        pair = (lambda q: _poisson_loss(case, q)) if case['eq'] == 'poisson' else \
            (lambda q: _stencil_loss(case, q))
    if case['call'] == 'train':
        if not wave:
            # a 32-bit run on differences over h^2 parts from a 64-bit one
            # within some hundred steps, whoever sums them
            return None
        w, m, v = [q.detach() for q in p], [0.0] * len(p), [0.0] * len(p)
        for k in range(1, case['epochs']):
            w = [q.requires_grad_() for q in w]
            loss = pair(w)[0]
            g = torch.autograd.grad(loss, w)
            done = [_adam(a.detach(), b, c, d, k) for a, b, c, d in zip(w, g, m, v)]
            w, m, v = (list(c) for c in zip(*done))
        return [loss.detach().reshape(1)] + w
    loss, norm = pair(p)
    g = torch.autograd.grad(loss, p)
    loss, norm = loss.detach(), norm.detach()
    if case['call'] == 'grad':
        return [loss.reshape(1), norm.reshape(1)] + list(g)
    shape = p[0].shape if wave else (-1,)
    flat = _flat(p).detach()
    m, v = _moments(flat.numel(), seed, _dtype(case))
    done = _adam(flat, _flat(g), m.double(), v.double(), DONE + 1)
    return [torch.stack([loss, norm])] + [c.reshape(shape) for c in done]
