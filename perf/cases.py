"""Performance cases of the quasistatic 3D xi step, through the public entry points.

Three kinds of case, each a dict of plain values:

* ``window``: consecutive xi steps of one time step's window
  (``PusherAndSolver3D.step_dt``: beam layer deposit, plasma step, beam move),
  started in the middle of the wake as a run started from a saved plasma state
  is, with an evolving particle beam or a rigid driver;
* ``deposit``, ``push``, ``solve``, ``filter``: one stage of the step through
  its own factory (``get_rhoj_computer``, ``get_plasma_particles_mover``,
  ``get_field_computer``, ``get_noise_filter``), as callers that assemble
  their own step use them.

Inputs are synthetic: the reference's particle lattice, displaced and set in
motion by a few smooth random modes of about a plasma wavelength plus thermal
noise, smooth fields, the charge and current density of those particles.
``exact`` restates each case in plain torch float64 (spline deposit and gather
by index_add and indexing, DST-I / DCT-I by torch.fft), following
plasma3d/move.py:28-148, weights.py:12-67, fields.py:112-322, solver.py:25-78,
noise_filter.py:53-238, beam3d/weights.py:40-64, beam3d/move.py:31-127 and
push_solver.py:215-286 of lcodePy.
"""
import math

import numpy as np
import torch

from lcodepy_amd.beam3d.beam_io import BeamDrain, BeamSource, RigidBeamDrain, RigidBeamSource
from lcodepy_amd.beam3d.data import BeamParticles
from lcodepy_amd.config import Config, good_size
from lcodepy_amd.plasma3d.data import Arrays
from lcodepy_amd.plasma3d.fields import get_field_computer
from lcodepy_amd.plasma3d.initialization import init_plasma
from lcodepy_amd.plasma3d.move import get_plasma_particles_mover
from lcodepy_amd.plasma3d.noise_filter import get_noise_filter
from lcodepy_amd.plasma3d.rhoj import get_rhoj_computer
from lcodepy_amd.push_solver import PusherAndSolver3D

FIELDS = ('Ex', 'Ey', 'Ez', 'Bx', 'By', 'Bz', 'Phi')
CURRENTS = ('ro', 'jx', 'jy', 'jz')
MOVING = ('x_offt', 'y_offt', 'px', 'py', 'pz', 'q')
PAD = 15            # cells between the plasma and the window edge (the default)
WALL = 10           # cells between the reflecting wall and the window edge
ION_MASS = 1836.0
F64 = torch.float64


# ---- the cases ----------------------------------------------------------------------
def _window(name, N, ppc, precision, steps, first=150, h=0.05, xi_step=0.02, beam=0,
            ions='background', solver='', pinch=0.0, **shape):
    return dict(name=name, kind='window', N=N, ppc=ppc, precision=precision, steps=steps,
                first=first, h=h, xi_step=xi_step, beam=beam, ions=ions, solver=solver,
                pinch=pinch, **shape)


def listed():
    return [
        # The smallest whole run: 129 x 129, 1 ppc, rigid driver, the config's
        # default field solver.  Launch latency and host work count.
        _window('rigid-129-fp64', 129, 1, 'fp64', 48, first=60, h=0.1, xi_step=0.05),
        # A member of a parameter scan: float32 bulk, rigid driver, LDS FFTs.
        _window('scan-257-fp32', 257, 1, 'fp32-bulk', 48, first=60, xi_step=0.05,
                solver='rfft'),
        # The size of the reference's own end-to-end tests: width 8, step
        # 0.05 -> 321 x 321, 4 ppc, an evolving beam of 1000 particles a layer.
        _window('evolve-321-fp64', 321, 4, 'fp64', 24, first=60, xi_step=0.05, beam=1000),
        # The benchmark workload near the driver's centre, both precision
        # forms: 513 x 513, 4 ppc, about 8000 beam particles a layer.  The
        # float32 form with its tuned FFT launch shape written into the
        # config, the float64 form tuned when the solver is built.
        _window('bench-513-fp32', 513, 4, 'fp32-bulk', 24, beam=8000, solver='rfft',
                rfft_cap=4096, rfft_tpb=2),
        _window('bench-513-fp64', 513, 4, 'fp64', 24, beam=8000, solver='auto'),
        # Two species: 769 x 769, 9 ppc, mobile ions, driver layers of 6000.
        _window('ions-769-fp64', 769, 9, 'fp64', 4, h=0.04, beam=6000, ions='mobile',
                solver='auto'),
        # The largest grid: 1025 x 1025, 4 ppc, float32 bulk, 20000 a layer.
        _window('large-1025-fp32', 1025, 4, 'fp32-bulk', 6, h=0.025, beam=20000, solver='rfft'),
        # Deposit where the wake's electrons cross: a pinched plasma with
        # cells of tens to hundreds of particles, odd grid, float32 bulk.
        dict(name='deposit-417-fp32', kind='deposit', N=417, ppc=4, precision='fp32-bulk',
             h=0.05, xi_step=0.02, ions='background', solver='rfft', pinch=0.85),
        # Push of a non-power-of-two window, float64.
        dict(name='push-385-fp64', kind='push', N=385, ppc=9, precision='fp64', h=0.05,
             xi_step=0.02, ions='background', solver='rfft', pinch=0.0),
        # Smallest and largest single field solves.
        dict(name='solve-65-fp64', kind='solve', N=65, ppc=1, precision='fp64', h=0.1,
             xi_step=0.05, ions='background', solver='', pinch=0.0),
        dict(name='solve-1025-fp64', kind='solve', N=1025, ppc=1, precision='fp64', h=0.025,
             xi_step=0.02, ions='background', solver='auto', pinch=0.0),
        # The declustering filter of a 449 x 449 window's lattice.
        dict(name='filter-449-fp64', kind='filter', N=449, ppc=4, precision='fp64', h=0.05,
             xi_step=0.02, ions='background', solver='rfft', pinch=0.0),
    ]


def _draw_N(rng, lo, hi):
    """A grid size the config accepts, spread over the logarithm of [lo, hi]."""
    want = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    sizes = [n for n in range(lo, hi + 1) if good_size(n)]
    return min(sizes, key=lambda n: abs(n - want))


def draw(rng):
    kind = rng.choice(['window', 'window', 'window', 'deposit', 'push', 'solve', 'filter'])
    precision = rng.choice(['fp64', 'fp32-bulk'])
    h = rng.choice([0.025, 0.04, 0.05, 0.1])
    xi_step = rng.choice([0.02, 0.05])
    solver = rng.choice(['rfft', 'rfft', ''])
    ions = rng.choice(['background', 'background', 'mobile'])
    pinch = rng.choice([0.0, 0.0, rng.uniform(0.3, 0.85)])
    if kind == 'window':
        N = _draw_N(rng, 65, 769 if solver else 513)
        ppc = rng.choice([1, 4, 9] if N <= 513 else [1, 4])
        cost = ppc * (N / 513) ** 2 * (2 if ions == 'mobile' else 1)
        steps = max(3, min(24, int(rng.uniform(24, 64) / max(cost, 1))))
        beam = rng.choice([0, int(math.exp(rng.uniform(math.log(200), math.log(20000))))])
        first = rng.randrange(int(3 / xi_step), int(6 / xi_step))
        case = _window('', N, ppc, precision, steps, first, h, xi_step, beam, ions, solver,
                       rng.choice([0.0, 0.0, rng.uniform(0.2, 0.6)]))
        del case['name']
        return case
    N = _draw_N(rng, 65, 1025 if kind == 'solve' and solver else 769)
    ppc = rng.choice([1, 4, 9, 16] if N <= 513 else [1, 4])
    return dict(kind=kind, N=N, ppc=ppc, precision=precision, h=h, xi_step=xi_step,
                ions='background' if kind == 'filter' else ions, solver=solver,
                pinch=pinch if kind == 'deposit' else 0.0)


def _config(case):
    N, h, s = case['N'], case['h'], case['xi_step']
    v = {'geometry': '3d', 'processing-unit-type': 'mi355x', 'precision': case['precision'],
         'window-width': (N - 1) * h / 2 + h / 2, 'transverse-step': h, 'xi-step': s,
         'window-length': (case.get('first', 0) + case.get('steps', 1) - 1) * s,
         'time-limit': 1.0, 'time-step': 1.0, 'ion-model': case['ions'], 'ion-mass': ION_MASS,
         'plasma-particles-per-cell': case['ppc'],
         'rigid-beam': case['kind'] == 'window' and not case['beam']}
    if case['solver']:
        v['field-solver'] = case['solver']
    for key in ('rfft_cap', 'rfft_tpb'):
        if case.get(key):
            v[key.replace('_', '-')] = case[key]
    if case['kind'] == 'filter':
        v['declustering-enabled'] = True
    config = Config(v)
    config._adjust_config_values_3d()
    assert config.getint('window-width-steps') == N
    return config


# ---- inputs, from the seed alone ---------------------------------------------------------
def _modes(rng, x, y, n=5, k=1.3):
    """A smooth random function of about unit size: n plane waves."""
    out = torch.zeros_like(x)
    for _ in range(n):
        kx, ky = rng.normal(0, k, 2)
        out += rng.normal(0, 1 / math.sqrt(n / 2)) * torch.cos(kx * x + ky * y
                                                                + rng.uniform(0, 2 * math.pi))
    return out


def _lattice(case):
    """The reference's lattice of round(sqrt(ppc))^2 particles a cell
    (plasma3d/initialization.py:72-135), x along the first index."""
    f = round(math.sqrt(case['ppc']))
    count = (case['N'] - 2 * PAD) // 2 * f
    ticks = torch.arange(count, dtype=F64, device='cuda')
    g = (torch.cat([-ticks[1:].flip(0), ticks]) if f % 2
         else torch.cat([-(ticks + 0.5).flip(0), ticks + 0.5])) * (case['h'] / f)
    n = len(g)
    return g[:, None].expand(n, n).contiguous(), g[None, :].expand(n, n).contiguous()


def _sort(case, rng, gen, ion):
    h, f = case['h'], round(math.sqrt(case['ppc']))
    bulk = (lambda a: a.float().double()) if case['precision'] == 'fp32-bulk' else (lambda a: a)
    x, y = _lattice(case)
    R = float(x.max()) + h
    edge = ((1 - (x / R) ** 2) * (1 - (y / R) ** 2)) ** 2
    heavy = ION_MASS if ion else 1.0
    r2 = x ** 2 + y ** 2
    squeeze = case['pinch'] * torch.exp(-r2 / (2 * (R / 4) ** 2))
    noise = [torch.randn(x.shape, dtype=F64, device='cuda', generator=gen) for _ in range(5)]
    dx = edge * (0.12 * _modes(rng, x, y) - squeeze * x + 2e-4 * noise[3]) / heavy
    dy = edge * (0.12 * _modes(rng, x, y) - squeeze * y + 2e-4 * noise[4]) / heavy
    ux = (edge * 0.15 * _modes(rng, x, y) + 1e-3 * noise[0]) / heavy
    uy = (edge * 0.15 * _modes(rng, x, y) + 1e-3 * noise[1]) / heavy
    uz = (ux ** 2 + uy ** 2) / 2 + (edge * 0.05 * _modes(rng, x, y) + 1e-3 * noise[2]) / heavy
    q = torch.full_like(x, (1.0 if ion else -1.0) / f ** 2 * h ** 2)
    m = torch.full_like(x, heavy / f ** 2 * h ** 2)
    return dict(x_init=x, y_init=y, x_offt=dx, y_offt=dy, px=bulk(m * ux), py=bulk(m * uy),
                pz=m * uz, q=bulk(q), m=bulk(m))


def _grid_xy(case):
    g = (torch.arange(case['N'], dtype=F64, device='cuda') - case['N'] // 2) * case['h']
    return torch.meshgrid(g, g, indexing='ij')


def _smooth_fields(case, rng, size):
    x, y = _grid_xy(case)
    R = case['N'] // 2 * case['h']
    edge = (1 - (x / R) ** 2) * (1 - (y / R) ** 2)
    return {k: (size * edge * _modes(rng, x, y)).contiguous() for k in FIELDS}


def _inputs(case, seed):
    """Everything of a case as float64 tensors (float32-rounded where the
    precision form stores float32)."""
    rng = np.random.RandomState(seed % (1 << 32))
    gen = torch.Generator(device='cuda')
    gen.manual_seed(seed)
    N, f32 = case['N'], case['precision'] == 'fp32-bulk'
    bulk = (lambda a: a.float().double()) if f32 else (lambda a: a)
    s = dict(fields=_smooth_fields(case, rng, 0.1))
    names = ('electrons', 'ions') if case['ions'] == 'mobile' else ('electrons',)
    s['sorts'] = {k: _sort(case, rng, gen, k == 'ions') for k in names}
    if case['kind'] in ('window', 'solve'):
        s['ro_initial'] = _ion_density(case)
        s['currents'] = {k: bulk(v) for k, v in
                         _currents(case, s['sorts'], s['ro_initial'], fixed=True).items()}
    if case['kind'] == 'solve':
        drift = {name: dict(a, x_offt=a['x_offt'] + a['px'] / a['m'] * case['xi_step'],
                            y_offt=a['y_offt'] + a['py'] / a['m'] * case['xi_step'])
                 for name, a in s['sorts'].items()}
        s['currents_full'] = {k: bulk(v) for k, v in
                              _currents(case, drift, s['ro_initial'], fixed=True).items()}
        s['rho_full'], s['rho_prev'] = (-0.3 * _gauss(case, d) for d in (0.0, 0.05))
    if case['kind'] == 'push':
        s['half'] = {k: bulk(v) for k, v in _smooth_fields(case, rng, 0.1).items()}
    if case['kind'] == 'window' and case['beam']:
        n, dxi = case['beam'] * case['steps'], case['xi_step']
        rand = lambda: torch.randn(n, dtype=F64, device='cuda', generator=gen)
        # Every layer holds case['beam'] particles, none within a thousandth of
        # a layer of its ends (where one of gamma 1000 could change layer).
        depth = torch.rand(case['steps'], case['beam'], dtype=F64, device='cuda', generator=gen)
        layer = case['first'] + torch.arange(case['steps'], device='cuda')
        xi = (-dxi * (layer[:, None] + 1e-3 + 0.998 * depth)).reshape(-1)
        sr = 0.08 * N * case['h'] / 2 if N * case['h'] < 12 else 0.5
        s['beam'] = dict(xi=xi.sort(descending=True).values, x=0.13 * sr + sr * rand(),
                         y=-0.07 * sr + sr * rand(), px=1e-2 * rand(), py=1e-2 * rand(),
                         pz=1000 + 10 * rand(), q_m=torch.full_like(xi, -1.0),
                         q_norm=torch.full_like(xi, -0.5 * 2 * math.pi * sr ** 2 / case['beam']))
    return s


def _gauss(case, shift):
    x, y = _grid_xy(case)
    return torch.exp(-((x - 0.2 - shift) ** 2 + (y + 0.1) ** 2) / 2).contiguous()


def _rigid_density(xp, xi, x, y):
    """A rigid driver, as a user writes one: a Gaussian, off the axis, its
    head at xi = 0 and its centre at xi = -3."""
    return -0.3 * xp.exp(-((x - 0.2) ** 2 + (y + 0.1) ** 2) / 2) * math.exp(-(xi + 3.0) ** 2 / 8)


# ---- what a user's program has in hand, and one pass ------------------------------------------
class _LastState:
    """Diagnostic that takes the state at the end of the window."""

    def after_step_dxi(self, *state):
        pass

    def dump(self, current_time, xi, particles, fields, currents, beam_drain):
        self.state = particles, fields, currents, beam_drain


def _wrap(group, like):
    return Arrays.wrap(**{k: v.to(getattr(like, k).dtype) for k, v in group.items()})


def prepare(case, seed):
    config = _config(case)
    s = _inputs(case, seed)
    state = dict(case=case, config=config)
    fields, particles, currents, const, _ = init_plasma(config)
    for name, a in s['sorts'].items():
        for k, v in a.items():
            t = getattr(particles[name], k)
            t.copy_(v.to(t.dtype))
    state.update(particles=particles, const=const, fields=_wrap(s['fields'], fields))
    kind = case['kind']
    if 'currents' in s:
        state['currents'] = _wrap(s['currents'], currents)
    if kind == 'window':
        state['solver'] = PusherAndSolver3D(config)
        state['solver'].verbose = False
        if case['beam']:
            b = s['beam']
            rows = [b[k] for k in ('xi', 'x', 'y', 'px', 'py', 'pz', 'q_m', 'q_norm')]
            ids = torch.arange(1, len(rows[0]) + 1, device='cuda')
            state['beam'] = BeamParticles(f=torch.stack(rows + [torch.zeros_like(rows[0])]),
                                          i=torch.stack([ids, torch.zeros_like(ids)]))
    elif kind == 'deposit':
        state['call'] = get_rhoj_computer(config)
    elif kind == 'push':
        state['call'] = get_plasma_particles_mover(config)
        half = torch.float32 if case['precision'] == 'fp32-bulk' else F64
        state['half'] = Arrays.wrap(**{k: v.to(half) for k, v in s['half'].items()})
    elif kind == 'solve':
        state['call'] = get_field_computer(config)
        state['currents_full'] = _wrap(s['currents_full'], currents)
        state['rho'] = s['rho_full'], s['rho_prev']
    elif kind == 'filter':
        state['call'] = get_noise_filter(config)
        # The filter kicks the particles of the new layer in place: their
        # momenta are taken from here on every pass.
        el = particles['electrons']
        state['kicked'] = Arrays.wrap(**{k: getattr(el, k) for k in el.names()
                                         if k not in ('px', 'py')})
    return state


def _out(group, keys):
    return {k: getattr(group, k) for k in keys}


def run(state):
    case, config = state['case'], state['config']
    kind, particles, const = case['kind'], state['particles'], state['const']
    if kind == 'window':
        last = _LastState()
        if case['beam']:
            source, drain = BeamSource(config, state['beam']), BeamDrain(config)
        else:
            source, drain = RigidBeamSource(config, _rigid_density), RigidBeamDrain(config)
        solver = state['solver']
        solver.step_dt(state['fields'], particles, state['currents'], const,
                       -(case['first'] - 1) * case['xi_step'], source, drain, 1.0, [last])
        particles, fields, currents, drain = last.state
        out = {name: _out(a, MOVING) for name, a in particles.items()}
        out.update(fields=_out(fields, FIELDS), currents=_out(currents, CURRENTS),
                   ez_axis=torch.stack(solver.ez_axis))
        if case['beam']:
            moved = drain.beam_slice()
            out['beam'] = _out(moved, ('xi', 'x', 'y', 'px', 'py', 'pz', 'id'))
        return out
    if kind == 'deposit':
        return _out(state['call'](particles, const), CURRENTS)
    if kind == 'push':
        free, smart = state['call']
        moved = smart(state['half'], particles, free(particles, const), const)
        return {name: _out(a, MOVING) for name, a in moved.items()}
    if kind == 'solve':
        full, half = state['call'](state['fields'], state['fields'], const, *state['rho'],
                                   state['currents'], state['currents_full'])
        return dict(full=_out(full, FIELDS), half=_out(half, FIELDS))
    kicked, el = state['kicked'], particles['electrons']
    kicked.px, kicked.py = el.px.clone(), el.py.clone()
    return _out(state['call'](kicked, el), ('px', 'py', 'dx_chaotic', 'dy_chaotic'))


# ---- what a pass cannot do without ------------------------------------------------------------
def work(case):
    N, kind = case['N'], case['kind']
    f = round(math.sqrt(case['ppc']))
    side = 2 * ((N - 2 * PAD) // 2 * f) - (f % 2)
    n, sorts = side * side, 2 if case['ions'] == 'mobile' else 1
    w = 4 if case['precision'] == 'fp32-bulk' else 8    # a bulk word
    # Particle state read (positions and pz float64; px py q m bulk) and
    # written (offsets and pz; px py q), a grid, and the operations of one
    # push, one deposit and one solve (paired complex FFTs of 2 (N - 1)).
    read, write, grid = 5 * 8 + 4 * w, 3 * 8 + 3 * w, N * N
    push, deposit = 25 * 12 + 150.0, 25 * 9 + 60.0
    length = 2 * (N - 1)
    solve = 7 * 4 * (N / 2) * 5 * length * math.log2(length) + 60 * grid
    if kind == 'window':
        step_bytes = n * sorts * (read + write) + grid * (14 * 8 + 16 * w + 16)
        step_flops = 3 * n * sorts * (push + deposit) + 2 * solve
        beam = case['beam']
        return dict(bytes=case['steps'] * (step_bytes + beam * 2 * 88),
                    flops=case['steps'] * (step_flops + beam * 900.0))
    if kind == 'deposit':
        return dict(bytes=n * sorts * read + 8 * grid * w, flops=n * sorts * deposit)
    if kind == 'push':
        return dict(bytes=n * sorts * (read + write) + 6 * grid * w, flops=n * sorts * push)
    if kind == 'solve':
        return dict(bytes=grid * (16 * w + 2 * 8 + 7 * 8 + 7 * 8 + 7 * w), flops=solve)
    return dict(bytes=n * (4 * 8 + 2 * 8 + 4 * w), flops=n * 150.0)


# ---- the same in plain torch, 64 bits -----------------------------------------------------------
def _weights(t):
    t2 = t * t
    return ((0.5 - t) ** 4 / 24,
            19 / 96 - 11 / 24 * t + t2 / 4 + t * t2 / 6 - t2 * t2 / 6,
            115 / 192 - 5 / 8 * t2 + t2 * t2 / 4,
            19 / 96 + 11 / 24 * t + t2 / 4 - t * t2 / 6 - t2 * t2 / 6,
            (0.5 + t) ** 4 / 24)


def _stencil(case, x, y):
    N, h = case['N'], case['h']
    xh, yh = x / h + 0.5, y / h + 0.5
    fx, fy = xh.floor(), yh.floor()
    cell = (fx + N // 2).long() * N + (fy + N // 2).long()
    return cell, _weights(xh - fx - 0.5), _weights(yh - fy - 0.5)


def _gamma(m, px, py, pz):
    return torch.sqrt(m * m + px * px + py * py + pz * pz)


FIXED = 2.0 ** 44   # units of the order-independent input densities


def _deposit(case, a, fixed=False):
    """(N, N, 4) density and currents of one sort; with ``fixed`` in integer
    units, so that the inputs made from it do not depend on the order of the
    additions."""
    N, h = case['N'], case['h']
    cols = [a[k].reshape(-1) for k in ('x_init', 'y_init', 'x_offt', 'y_offt', 'px', 'py', 'pz',
                                       'q', 'm')]
    x_init, y_init, x_offt, y_offt, px, py, pz, q, m = cols
    cell, wx, wy = _stencil(case, x_init + x_offt, y_init + y_offt)
    gamma = _gamma(m, px, py, pz)
    ro = q / (1 - pz / gamma) / h ** 2
    c = torch.stack([ro, ro * px / gamma, ro * py / gamma, ro * pz / gamma], 1)
    out = torch.zeros(N * N, 4, dtype=torch.int64 if fixed else F64, device='cuda')
    for i in range(5):
        for j in range(5):
            v = c * (wx[i] * wy[j])[:, None]
            out.index_add_(0, cell + ((i - 2) * N + j - 2),
                           (v * FIXED).round().long() if fixed else v)
    return (out.double() / FIXED if fixed else out).reshape(N, N, 4)


def _ion_density(case):
    x, y = _lattice(case)
    z = torch.zeros_like(x)
    f = round(math.sqrt(case['ppc']))
    q = torch.full_like(x, 1.0 / f ** 2 * case['h'] ** 2)
    rest = dict(x_init=x, y_init=y, x_offt=z, y_offt=z, px=z, py=z, pz=z, q=q, m=q)
    return _deposit(case, rest, fixed=True)[..., 0].contiguous()


def _currents(case, sorts, ro_initial, fixed=False):
    N = case['N']
    out = {k: torch.zeros(2, N, N, dtype=F64, device='cuda') for k in CURRENTS}
    for column, a in enumerate(sorts.values()):
        d = _deposit(case, a, fixed)
        for i, k in enumerate(CURRENTS):
            out[k][column] = d[..., i]
    if case['ions'] == 'background' and ro_initial is not None:
        out['ro'][1] = ro_initial
    return out


def _reflect(init, pos, offt, b):
    up, down = pos > b, pos < -b
    pos = torch.where(up, 2 * b - pos, torch.where(down, -2 * b - pos, pos))
    return pos, torch.where(up | down, pos - init, offt), up | down


def _free(case, a):
    d = _gamma(a['m'], a['px'], a['py'], a['pz']) - a['pz']
    return dict(a, x_offt=a['x_offt'] + a['px'] / d * case['xi_step'],
                y_offt=a['y_offt'] + a['py'] / d * case['xi_step'])


def _push(case, fields, prev, est):
    """Smart push of one sort from layer k (prev) with the estimate est."""
    dxi, N = case['xi_step'], case['N']
    b = case['h'] * (N / 2 - WALL)
    xi0, yi0, m, q = prev['x_init'], prev['y_init'], prev['m'], est['q']
    xop, yop, opx, opy, opz = (prev[k] for k in ('x_offt', 'y_offt', 'px', 'py', 'pz'))
    x, _, hx = _reflect(xi0, xi0 + (xop + est['x_offt']) / 2, xop, b)
    y, _, hy = _reflect(yi0, yi0 + (yop + est['y_offt']) / 2, yop, b)
    zero = torch.zeros_like(x)
    hit = hx | hy
    px, py, pz = (torch.where(hit, zero, v) for v in (opx, opy, opz))
    cell, wx, wy = _stencil(case, x, y)
    F = {k: torch.zeros_like(x) for k in FIELDS[:6]}
    flat = {k: fields[k].reshape(-1) for k in F}
    for i in range(5):
        for j in range(5):
            w, o = wx[i] * wy[j], cell + ((i - 2) * N + j - 2)
            for k in F:
                F[k] += flat[k][o] * w
    for _ in range(2):
        gamma = _gamma(m, px, py, pz)
        vx, vy, vz = px / gamma, py / gamma, pz / gamma
        factor = q * dxi / (1 - vz)
        dpx = factor * (F['Ex'] + vy * F['Bz'] - vz * F['By'])
        dpy = factor * (F['Ey'] - vx * F['Bz'] + vz * F['Bx'])
        dpz = factor * (F['Ez'] + vx * F['By'] - vy * F['Bx'])
        px, py, pz = opx + dpx / 2, opy + dpy / 2, opz + dpz / 2
    d = _gamma(m, px, py, pz) - pz
    xo, yo = xop + px / d * dxi, yop + py / d * dxi
    px, py, pz = opx + dpx, opy + dpy, opz + dpz
    x, xo, hx = _reflect(xi0, xi0 + xo, xo, b)
    y, yo, hy = _reflect(yi0, yi0 + yo, yo, b)
    hit = hx | hy
    x, y = xi0 + xo, yi0 + yo
    gone = (x >= b) | (x <= -b) | (y >= b) | (y <= -b)
    px, py, pz = (torch.where(hit | gone, zero, v) for v in (px, py, pz))
    new = dict(x_offt=torch.where(gone, zero, xo), y_offt=torch.where(gone, zero, yo), px=px,
               py=py, pz=pz, q=torch.where(gone, zero, q))
    return {**est, **{k: torch.where(q == 0, est[k], v) for k, v in new.items()}}


def _cosine(a, dim):
    """DCT-I along dim."""
    inner = a.narrow(dim, 1, a.shape[dim] - 2)
    return torch.fft.rfft(torch.cat([a, inner.flip(dim)], dim), dim=dim).real


def _sine(a, dim):
    """DST-I along dim of the inner points; the edge points are zero."""
    inner = a.narrow(dim, 1, a.shape[dim] - 2)
    edge = torch.zeros_like(a.narrow(dim, 0, 1))
    return -torch.fft.rfft(torch.cat([edge, inner, edge, -inner.flip(dim)], dim), dim=dim).imag


def _invert(case, rhs, sine_x, sine_y, c):
    N, h = case['N'], case['h']
    lam = 4 / h ** 2 * torch.sin(torch.arange(N, dtype=F64, device='cuda')
                                 * math.pi / (2 * (N - 1))) ** 2
    both = lam[:, None] + lam[None, :] + c
    scale = torch.where(both > 0, 1 / both, torch.zeros_like(both)) / (2 * (N - 1)) ** 2
    tx, ty = (_sine if s else _cosine for s in (sine_x, sine_y))
    return ty(tx(scale * tx(ty(rhs, 1), 0), 0), 1)


def _slope(a, dim):
    out = torch.zeros_like(a)
    inner = (a[2:, 1:-1] - a[:-2, 1:-1]) if dim == 0 else (a[1:-1, 2:] - a[1:-1, :-2])
    out[1:-1, 1:-1] = inner
    return out


def _solve(case, pred, prev, rho_full, rho_prev, cur_prev, cur_full, c):
    """(fields_full, fields_half) of one solve."""
    h, dxi = case['h'], case['xi_step']
    f = {k: v.sum(0) for k, v in cur_full.items()}
    p = {k: v.sum(0) for k, v in cur_prev.items()}
    ro = (f['ro'] + rho_full + p['ro'] + rho_prev) / 2
    jz = (f['jz'] + rho_full + p['jz'] + rho_prev) / 2
    djx, djy = (p['jx'] - f['jx']) / dxi, (p['jy'] - f['jy']) / dxi
    s = 1 / (2 * h)
    half = dict(
        Ex=_invert(case, -(_slope(ro, 0) * s - djx - c * pred['Ex']), False, True, c),
        Ey=_invert(case, -(_slope(ro, 1) * s - djy - c * pred['Ey']), True, False, c),
        Bx=_invert(case, _slope(jz, 1) * s - djy + c * pred['Bx'], True, False, c),
        By=_invert(case, -(_slope(jz, 0) * s - djx - c * pred['By']), False, True, c))
    full = {k: 2 * v - prev[k] for k, v in half.items()}
    full['Ez'] = _invert(case, -(_slope(f['jx'], 0) + _slope(f['jy'], 1)) * s, True, True, 0.0)
    bz = _invert(case, -(_slope(f['jx'], 1) - _slope(f['jy'], 0)) * s, False, False, 0.0)
    full['Bz'] = bz - bz.mean()
    full['Phi'] = half['Phi'] = _invert(case, f['ro'] - f['jz'], True, True, 0.0)
    for k in ('Ez', 'Bz'):
        half[k] = (full[k] + prev[k]) / 2
    return full, half


def _coefficient(case):
    """The solver's subtraction coefficient: the default '1' becomes 1 + xi_step."""
    return 1 + case['xi_step']


def _step(case, sorts, fields, cur, ro_initial, rho_full, rho_prev):
    c = _coefficient(case)
    new = {k: _push(case, fields, a, _free(case, a)) for k, a in sorts.items()}
    cf = _currents(case, new, ro_initial)
    _, half = _solve(case, fields, fields, rho_full, rho_prev, cur, cf, c)
    new = {k: _push(case, half, sorts[k], a) for k, a in new.items()}
    cf = _currents(case, new, ro_initial)
    full, half = _solve(case, half, fields, rho_full, rho_prev, cur, cf, c)
    new = {k: _push(case, half, sorts[k], a) for k, a in new.items()}
    return new, full, _currents(case, new, ro_initial)


def _beam_deposit(case, layer, index, running, following):
    N, dxi = case['N'], case['xi_step']
    cell, wx, wy = _stencil(case, layer['x'], layer['y'])
    share = (-dxi * index - layer['xi']) / dxi
    for i in range(5):
        for j in range(5):
            w, o = layer['q_norm'] * (wx[i] * wy[j]), cell + ((i - 2) * N + j - 2)
            running.view(-1).index_add_(0, o, w * share)
            following.view(-1).index_add_(0, o, w * (1 - share))


def _beam_move(case, b, index, fk, fk1):
    """One move of a layer whose particles take whole time steps (gamma about
    1000): 'left' counts the steps they still have to take.  Returns the
    moved and the fell particles."""
    N, h, dxi = case['N'], case['h'], case['xi_step']
    xi_k, xi_k1 = -(index - 1) * dxi, -index * dxi
    wide = h * N / 2
    r2 = max(0.9 * wide, wide - 1) ** 2
    d = 1.0
    X, Y, XI, PX, PY, PZ = (b[k] for k in ('x', 'y', 'xi', 'px', 'py', 'pz'))
    gamma = torch.sqrt(1 + PX ** 2 + PY ** 2 + PZ ** 2)
    xh, yh, xih = X + d / 2 * PX / gamma, Y + d / 2 * PY / gamma, XI + d / 2 * (PZ / gamma - 1)
    go = b['left'] > 0
    drops = go & (xi_k1 > xih)
    lost = go & ~drops & (xh ** 2 + yh ** 2 >= r2)
    cell, wx, wy = _stencil(case, xh, yh)
    cell = cell.clamp(2 * N + 2, N * N - 2 * N - 3)
    share = (xih - xi_k) / dxi
    F = {k: torch.zeros_like(X) for k in FIELDS[:6]}
    for i in range(5):
        for j in range(5):
            w, o = wx[i] * wy[j], cell + ((i - 2) * N + j - 2)
            for k in F:
                F[k] += (fk[k].reshape(-1)[o] * share + fk1[k].reshape(-1)[o] * (1 - share)) * w
    vx, vy, vz = PX / gamma, PY / gamma, PZ / gamma
    hx = PX - d / 2 * (F['Ex'] + vy * F['Bz'] - vz * F['By'])
    hy = PY - d / 2 * (F['Ey'] + vz * F['Bx'] - vx * F['Bz'])
    hz = PZ - d / 2 * (F['Ez'] + vx * F['By'] - vy * F['Bx'])
    gamma = torch.sqrt(1 + hx ** 2 + hy ** 2 + hz ** 2)
    new = dict(x=X + d * hx / gamma, y=Y + d * hy / gamma, xi=XI + d * (hz / gamma - 1),
               px=2 * hx - PX, py=2 * hy - PY, pz=2 * hz - PZ, left=b['left'] - 1)
    done = go & ~drops & ~lost
    lost |= done & (new['x'] ** 2 + new['y'] ** 2 >= r2)
    out = {**b, **{k: torch.where(done, v, b[k]) for k, v in new.items()}}
    # A particle that has no step left falls by its x, as move.py:123 has it.
    fell = drops | ((out['left'] == 0) & (xi_k1 > out['x']))
    take = lambda keep: {k: v[keep] for k, v in out.items()}
    return take(~fell & ~lost), take(fell)


def _join(groups):
    return {k: torch.cat([g[k] for g in groups]) for k in groups[0]}


def _exact_window(case, s):
    N, dxi, h = case['N'], case['xi_step'], case['h']
    sorts, fields, cur = s['sorts'], s['fields'], s['currents']
    grid = lambda: torch.zeros(N, N, dtype=F64, device='cuda')
    rho_prev, running, ez = grid(), grid(), []
    drained, fell, last = [], None, None
    if case['beam']:
        beam = dict(s['beam'])
        beam['id'] = torch.arange(1, len(beam['x']) + 1, device='cuda')
        beam['left'] = torch.zeros_like(beam['id'])
    else:
        g = (torch.arange(N, dtype=F64, device='cuda') - N // 2) * h
        x, y = torch.meshgrid(g, g, indexing='xy')
    for i in range(case['first'], case['first'] + case['steps']):
        if case['beam']:
            here = (beam['xi'] < -dxi * i) & (beam['xi'] >= -dxi * (i + 1))
            layer = {k: v[here] for k, v in beam.items()}
            following = grid()
            _beam_deposit(case, layer, i, running, following)
            rho, running = running / h ** 2, following
        else:
            rho = _rigid_density(torch, -i * dxi, x, y)
        before = fields
        sorts, fields, cur = _step(case, sorts, fields, cur, s['ro_initial'], rho, rho_prev)
        if case['beam']:
            if last is not None:
                last['left'] = torch.ones_like(last['left'])
                moving = last if fell is None else _join([last, fell])
                moved, fell = _beam_move(case, moving, i, before, fields)
                drained.append(moved)
            last = layer
        rho_prev = rho
        ez.append(fields['Ez'][N // 2, N // 2])
    out = {name: {k: a[k] for k in MOVING} for name, a in sorts.items()}
    out.update(fields=fields, currents=cur, ez_axis=torch.stack(ez))
    if case['beam']:
        out['beam'] = {k: _join(drained)[k] for k in ('xi', 'x', 'y', 'px', 'py', 'pz')}
        out['beam']['id'] = None
    return out


def _inhomogeneity(d, dim):
    a = d if dim else d.T
    out = torch.zeros_like(a)
    l, c, r = a[:, :-2], a[:, 1:-1], a[:, 2:]
    zero = torch.zeros_like(c)
    out[:, 1:-1] = torch.where((l != 0) & (c != 0) & (r != 0), c - (l + r) / 2, zero)
    for at, o in ((0, (0, 1, 2)), (-1, (-1, -2, -3))):
        u, v, w = (a[:, k] for k in o)
        out[:, at] = torch.where((u != 0) & (v != 0) & (w != 0), u - 2 * v + w, zero[:, 0])
    return out if dim else out.T


def _exact_filter(case, a):
    """The declustering filter with the config's defaults (averaging 3, force
    0.3, limit 1e-3, no damping: its key is read under another spelling)."""
    n = len(a['x_offt'])
    k = torch.fft.fftfreq(n, dtype=F64, device='cuda')
    g = torch.exp(-2 * math.pi ** 2 * 3.0 ** 2 * k ** 2)
    smooth = lambda v: torch.fft.ifft2(torch.fft.fft2(v) * (g[:, None] * g[None, :])).real
    chaotic = []
    for d in (a['x_offt'], a['y_offt']):
        i = (_inhomogeneity(d, 0) + _inhomogeneity(d, 1)) / 2
        chaotic.append(i - smooth(i))
    dist = chaotic[0] ** 2 + chaotic[1] ** 2
    near = torch.where(dist < 1e-3 ** 2, 1 - dist / 1e-3 ** 2, torch.zeros_like(dist))
    out = {}
    for key, c in (('px', chaotic[0]), ('py', chaotic[1])):
        force, p = -0.3 * c * near, a[key].clone()
        for p_, f in ((p, force), (p.T, force.T)):
            p_[1:-1] += case['xi_step'] * f[1:-1] / 2
            p_[2:] -= case['xi_step'] * f[1:-1] / 4
            p_[:-2] -= case['xi_step'] * f[1:-1] / 4
        out[key] = p
    return dict(out, dx_chaotic=chaotic[0], dy_chaotic=chaotic[1])


def exact(case, seed):
    s = _inputs(case, seed)
    kind = case['kind']
    if kind == 'window':
        return _exact_window(case, s)
    if kind == 'deposit':
        return _currents(case, s['sorts'], _ion_density(case))
    if kind == 'push':
        return {name: {k: v for k, v in _push(case, s['half'], a, _free(case, a)).items()
                       if k in MOVING} for name, a in s['sorts'].items()}
    if kind == 'solve':
        full, half = _solve(case, s['fields'], s['fields'], s['rho_full'], s['rho_prev'],
                            s['currents'], s['currents_full'], _coefficient(case))
        return dict(full=full, half=half)
    return _exact_filter(case, s['sorts']['electrons'])
