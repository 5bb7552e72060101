"""The work that users of this framework have it do, as timed cases.

Each case goes through the public entry points: the scattering-model plugins
(``fs`` for one spatial DOF, ``fs_batch`` for a bank), the collision system
with FR advection, and the learned stand-in's forward pass and training
gradient.  ``listed`` holds the cases, ``draw`` gives more of the same ranges,
``prepare`` makes what a program holds before the call, ``run`` is one pass,
``work`` the bytes and flops a pass cannot do without, and ``exact`` the same
outputs from plain torch and NumPy in 64 bits (for the operator the formula as
it is published: one transform pair per radial node and direction).

A case's ``op`` is one of
  fs       one DOF through the per-DOF plugin call
  batch    a whole bank through ``fs_batch`` (model vhs, nodal or vss)
  rhs      Q plus FR advection of a bank on a periodic quad mesh
  forward  the learned stand-in's network on normalised rows
  gradient the training gradient of one mini-batch
"""
import functools
import glob
import math
import os
import re

import numpy as np
import torch

import frfs_amd

ARGON = dict(T0=273.0, H0=1e-3, rho0=0.00011140244750324529, molarMass0=39.96e-3)
GAS_R, AVOGADRO = 8.3144598, 6.0221409e+23
DESIGNS = os.path.join(os.path.dirname(os.path.abspath(frfs_amd.__file__)), 'sphericaldesign', 'symmetric')
D_REF, T_REF, DEV = 4.17e-10, 273.0, {8: 5.0, 16: 5.0, 24: 5.5, 32: 6.0}
MPRE = 32
SECOND_MASS = 2 * 39.96e-3
F_REF = math.pi ** -1.5
WIDTH, MODES = 32, 8


def listed():
    vss = dict(op='batch', model='vss', Nv=32, Nrho=16, M=12, species=1)
    return [
        # the plugin's per-DOF call, the way a solver's own DOF loop makes it
        dict(vss, name='fs_vss32_mixed', op='fs', nupts=4, neles=40, precision='mixed', project=1),
        # the smallest whole problem: 64 homogeneous DOFs, hard spheres, the default precision
        dict(name='vhs16_double', op='batch', model='vhs', Nv=16, Nrho=8, M=6, species=1, nupts=1, neles=64,
             precision='double', project=0),
        # teacher of the learned stand-in: one chunk of training targets (projected FP64)
        dict(name='vhs16_double_targets', op='batch', model='vhs', Nv=16, Nrho=8, M=6, species=1, nupts=1, neles=8192,
             precision='double', project=1),
        # bilinear Q(f, g) of the nodal plugin, a small odd mesh of p = 2 quads
        dict(name='nodal24_double', op='batch', model='nodal', Nv=24, Nrho=8, M=6, species=1, nupts=9, neles=11,
             precision='double', project=0),
        # a velocity grid without kernels of its own
        dict(name='vhs20_double', op='batch', model='vhs', Nv=20, Nrho=10, M=6, species=1, nupts=9, neles=17,
             precision='double', project=0),
        # the default precision on the large grid: a modest mesh of p = 1 quads
        dict(vss, name='vss32_double', nupts=4, neles=128, precision='double', project=0),
        # the same at full size in mixed precision with the projection, the schedule the tuner picks
        dict(vss, name='vss32_mixed', nupts=1, neles=4096, precision='mixed', project=1, max_chunk=2048, accum_quad=1),
        # a binary mixture (mass ratio 1:2), ragged bank
        dict(vss, name='vss32_two_species', species=2, nupts=4, neles=75, precision='mixed', project=1),
        # right-hand side of a solver stage: collisions and advection on a 32 x 32 mesh of p = 2 quads
        dict(name='rhs24_mixed', op='rhs', model='vhs', Nv=24, Nrho=12, M=6, species=1, nelx=32, nely=32, order=2,
             precision='mixed', project=1),
        # the stand-in at inference: a full chunk on the small grid, a ragged one on the large grid
        dict(name='fno16_forward', op='forward', Nv=16, layers=4, rows=8192),
        dict(name='fno32_forward', op='forward', Nv=32, layers=4, rows=700),
        # the stand-in in training: one mini-batch with the conservation penalty
        dict(name='fno16_gradient', op='gradient', Nv=16, layers=4, rows=64),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(['fs', 'vhs', 'vhs', 'nodal', 'other_grid', 'vss', 'vss', 'mixture', 'rhs', 'forward', 'gradient'])
    precision = rng.choice(['double', 'mixed'])
    project = rng.choice([0, 1])
    nupts = rng.choice([1, 3, 4, 9])

    def bank(most):
        d = _log_int(rng, 1, most)
        return dict(nupts=nupts, neles=max(1, d // nupts))

    if kind == 'fs':
        if rng.random() < 0.5:
            m = dict(model='vss', Nv=32, Nrho=rng.choice([8, 12, 16]), M=12)
        else:
            m = dict(model='vhs', Nv=rng.choice([16, 24]), Nrho=8, M=6)
        return dict(m, op='fs', species=1, nupts=nupts, neles=rng.randint(1, 80), precision=precision, project=project)
    if kind == 'vhs':
        nv = rng.choice([8, 16, 16, 24])
        return dict(bank({8: 16384, 16: 8192, 24: 2048}[nv]), op='batch', model='vhs', Nv=nv, Nrho=rng.choice([6, 8, 12]), M=6,
                    species=1, precision=precision, project=project)
    if kind == 'nodal':
        nv = rng.choice([8, 16, 24])
        return dict(bank({8: 4096, 16: 1024, 24: 300}[nv]), op='batch', model='nodal', Nv=nv, Nrho=rng.choice([4, 8]), M=6,
                    species=1, precision=precision, project=project)
    if kind == 'other_grid':
        nv = rng.choice([10, 12, 14, 18, 20, 22, 28, 36, 40, 48])
        return dict(bank(max(2, int(180 * (20.0 / nv) ** 3))), op='batch', model='vhs', Nv=nv, Nrho=rng.choice([6, 8, 10]), M=6,
                    species=1, precision=precision, project=project)
    if kind == 'vss':
        nv = rng.choice([16, 24, 32, 32])
        return dict(bank({16: 2048, 24: 768, 32: 512}[nv]), op='batch', model='vss', Nv=nv, Nrho=rng.choice([6, 8, 16]), M=12,
                    species=1, precision=precision, project=project)
    if kind == 'mixture':
        nv = rng.choice([16, 32])
        return dict(bank({16: 800, 32: 200}[nv]), op='batch', model='vss', Nv=nv, Nrho=rng.choice([6, 8, 16]), M=12, species=2,
                    precision=precision, project=project)
    if kind == 'rhs':
        order = rng.choice([1, 2, 3])
        return dict(op='rhs', model='vhs', Nv=rng.choice([16, 24]), Nrho=8, M=6, species=1, nelx=rng.randint(2, 24),
                    nely=rng.randint(2, 24), order=order, precision=precision, project=project)
    nv = rng.choice([16, 32])
    if kind == 'forward':
        return dict(op='forward', Nv=nv, layers=rng.choice([2, 3, 4, 4, 6]), rows=_log_int(rng, 1, 8192 if nv == 16 else 1024))
    return dict(op='gradient', Nv=nv, layers=rng.choice([2, 4]), rows=_log_int(rng, 4, 256 if nv == 16 else 64))


# ---------------------------------------------------------------- the case in plain numbers
def _dev(c):
    return DEV.get(c['Nv'], 5.0)


def _masses(c):
    return [ARGON['molarMass0'], SECOND_MASS][:c['species']]


def _points(c):
    """Solution points per element and elements of the case's bank."""
    return ((c['order'] + 1) ** 2, c['nelx'] * c['nely']) if c['op'] == 'rhs' else (c['nupts'], c['neles'])


def _config(c):
    from frfs_amd.inifile import Inifile
    sm = {'type': {'vhs': 'vhs-gll', 'nodal': 'vhs-gll-nodal', 'vss': 'vss-gll'}[c['model']],
          'precision': c['precision'], 'conservation-projection': c['project'],
          'max-chunk': c.get('max_chunk', 0), 'accum-quad': c.get('accum_quad', 0)}
    mesh = {'dev': _dev(c), 'cmax': 0, 'Tmax': 273}
    if c['model'] == 'vss':
        sm |= {'ssrulepre': 'womersley', 'Mpre': MPRE}
        for pq, (alpha, omega, dref, tref) in _pairs(c).items():
            sm |= {'alpha' + pq: alpha, 'omega' + pq: omega, 'dRef' + pq: dref, 'Tref' + pq: tref}
        mesh |= {'molarMass%d' % (p + 1): m for p, m in enumerate(_masses(c))}
    else:
        sm |= {'omega': 0.5, 'dRef': D_REF, 'Tref': T_REF}
    return Inifile.from_dict({
        'non-dim': ARGON, 'constants': {'Nv': c['Nv'], 'NvBatchSize': c['Nv'] ** 3, 'Nrho': c['Nrho']},
        'velocity-mesh': mesh, 'spherical-design-rule': {'ssrule': 'womersley', 'M': c['M']}, 'scattering-model': sm})


def _pairs(c):
    """(alpha, omega, dRef, Tref) of every species pair."""
    omega, size = (0.74, 0.81), (1.0, 1.3)
    return {'%d%d' % (p, q): (1.4, 0.5 * (omega[p] + omega[q]), 0.5 * (size[p] + size[q]) * D_REF, T_REF)
            for p in range(c['species']) for q in range(c['species'])}


def _nodes(n):
    x = np.linspace(-1, 1, 2 * n + 1)[1::2] * _half_width(n)
    return x


def _half_width(n):
    return DEV.get(n, 5.0)


def _grid(n):
    """Velocity coordinates (3, n^3) on the box of the case's grid."""
    x = _nodes(n)
    return np.stack([a.reshape(-1) for a in np.meshgrid(x, x, x, indexing='ij')])


def _device():
    return 'cuda' if torch.cuda.is_available() else 'cpu'


# ---------------------------------------------------------------- inputs, from the seed alone
def _mixture(cv, par, mass=1.0):
    """Rows of f = sum_k n_k (m / (pi T_k))^1.5 exp(-m |c - u_k|^2 / T_k); par (rows, components, 5)."""
    c = torch.as_tensor(cv, dtype=torch.float64, device=_device())
    par = torch.as_tensor(par, dtype=torch.float64, device=_device())
    out = torch.empty((par.shape[0], c.shape[1]), dtype=torch.float64, device=_device())
    for b in range(0, par.shape[0], 256):
        acc = 0
        for k in range(par.shape[1]):
            n, u, t = par[b:b + 256, k, 0:1], par[b:b + 256, k, 1:4], par[b:b + 256, k, 4:5]
            r2 = (c[0] - u[:, 0:1]) ** 2 + (c[1] - u[:, 1:2]) ** 2 + (c[2] - u[:, 2:3]) ** 2
            acc = acc + n * (mass / (math.pi * t)) ** 1.5 * torch.exp(-mass * r2 / t)
        out[b:b + 256] = acc
    return out


def _two_maxwellians(rows, rng):
    """Seeded two-component states: n ~ U(0.5, 1.5), u ~ U(-1, 1)^3, T ~ U(0.5, 2) each."""
    return np.concatenate([rng.uniform(0.5, 1.5, (rows, 2, 1)), rng.uniform(-1, 1, (rows, 2, 3)),
                           rng.uniform(0.5, 2, (rows, 2, 1))], axis=2)


def _shear_layer(c, rng):
    """A smooth two-component flow on the periodic mesh, one row per (element, point)."""
    x = np.polynomial.legendre.leggauss(c['order'] + 1)[0]
    ex, ey = np.arange(c['nelx']), np.arange(c['nely'])
    px = ((ex[:, None] + 0.5 * (x + 1)) / c['nelx'])[None, :, None, :]
    py = ((ey[:, None] + 0.5 * (x + 1)) / c['nely'])[:, None, :, None]
    px, py = (np.broadcast_to(a, (c['nely'], c['nelx'], x.size, x.size)).reshape(-1) for a in (px, py))
    wave = lambda: np.sin(2 * math.pi * (rng.integers(1, 3) * px + rng.integers(0, 3) * py + rng.uniform()))  # noqa: E731
    par = np.empty((px.size, 2, 5))
    for k, share in enumerate((0.8, 0.3)):
        par[:, k, 0] = share * (1 + 0.2 * wave())
        for d in range(3):
            par[:, k, 1 + d] = rng.uniform(-0.4, 0.4) + 0.3 * wave()
        par[:, k, 4] = rng.uniform(0.8, 1.3) + 0.2 * wave()
    return par


def _rows(c, seed):
    """The input distributions of a collision case: one (rows, Nv^3) tensor per source."""
    rng = np.random.default_rng([seed, 11])
    cv = _grid(c['Nv'])
    nupts, neles = _points(c)
    if c['op'] == 'rhs':
        return [_mixture(cv, _shear_layer(c, rng))]
    if c['model'] == 'nodal':
        return [_mixture(cv, _two_maxwellians(nupts * neles, rng)) for _ in range(2)]
    out = []
    for s in range(c['species']):
        par = _two_maxwellians(nupts * neles, rng)
        if c['species'] > 1:
            par[:, :, 0] *= 0.4 + 0.3 * s
        out.append(_mixture(cv, par, mass=_masses(c)[s] / ARGON['molarMass0']))
    return out


def _to_bank(rows, nupts, neles):
    """(neles * nupts, n) rows in the banks' layout: 32 elements of a point and velocity side by side."""
    n, pad = rows.shape[1], -(-neles // 32) * 32
    a = rows.new_zeros((nupts, n, pad))
    a[..., :neles] = rows.reshape(neles, nupts, n).permute(1, 2, 0)
    return a.reshape(nupts, n, pad // 32, 32).permute(0, 2, 1, 3).reshape(-1).contiguous()


def _theta(layers, seed):
    """Seeded network weights in the flat layout of the stand-in: lift (P, p0), per layer the mode
    weights (in, out, mode, re/im), the pointwise matrix (out, in) and bias, then the projection."""
    rng = np.random.default_rng([seed, 13])
    lim, parts = 1 / math.sqrt(WIDTH), [rng.uniform(-1, 1, WIDTH), rng.uniform(-0.1, 0.1, WIDTH)]
    for _ in range(layers):
        parts += [rng.uniform(-1, 1, 2 * WIDTH * WIDTH * MODES ** 3) / WIDTH ** 1.5, rng.uniform(-lim, lim, WIDTH * WIDTH),
                  rng.uniform(-lim, lim, WIDTH)]
    return np.concatenate(parts + [rng.uniform(-lim, lim, WIDTH), np.zeros(1)]).astype(np.float32)


def _training_rows(c, seed):
    """Normalised rows g = f / (rho f_ref) and targets of unit RMS (the relaxation towards the local Maxwellian)."""
    rng = np.random.default_rng([seed, 17])
    cv, cw = _grid(c['Nv']), (2 * _half_width(c['Nv']) / c['Nv']) ** 3
    par = _two_maxwellians(c['rows'], rng)
    f = _mixture(cv, par)
    g = (f / (f.sum(1, keepdim=True) * cw * F_REF)).float()
    if c['op'] == 'forward':
        return g, None
    n, u, t = par[..., 0:1], par[..., 1:4], par[..., 4:5]
    rho = n.sum(1, keepdims=True)
    um = (n * u).sum(1, keepdims=True) / rho
    tm = (n * (t + 2 / 3 * ((u - um) ** 2).sum(2, keepdims=True))).sum(1, keepdims=True) / rho
    q = _mixture(cv, np.concatenate([np.ones_like(rho), um, tm], axis=2)) - f / torch.as_tensor(rho[:, 0], device=f.device)
    return g, (q / q.square().mean().sqrt()).float()


# ---------------------------------------------------------------- the framework's side
def prepare(case, seed):
    from frfs_amd.backend import HIPBackend
    c = case
    be = HIPBackend()
    if c['op'] in ('forward', 'gradient'):
        from frfs_amd.surrogate import FourierSurrogate, gram
        net = FourierSurrogate(be, layers=c['layers'], theta=_theta(c['layers'], seed), nv=c['Nv'])
        g, t = _training_rows(c, seed)
        if c['op'] == 'gradient':
            half, n = _half_width(c['Nv']), c['Nv']
            cw = (2 * half / n) ** 3
            net.cons_weight, net.cons = 10.0, (half, cw, torch.tensor(gram(_grid(n), cw)[0].reshape(-1), device=be.device))
            return dict(op='gradient', net=net, g=g, t=t)
        return dict(op='forward', net=net, g=g, out=torch.empty_like(g))
    rows = _rows(c, seed)
    nupts, neles = _points(c)
    shape = (nupts, c['Nv'] ** 3, neles)
    if c['op'] == 'rhs':
        from frfs_amd.fr import PeriodicQuadAdvection
        from frfs_amd.system import DGFSCollisionSystem
        s = DGFSCollisionSystem(be, _config(c), nupts, neles)
        adv = PeriodicQuadAdvection(be, s.vm, c['nelx'], c['nely'], 1.0 / c['nelx'], 1.0 / c['nely'], order=c['order'])
        s.rhs = lambda t, uin, fout: adv(s.banks[uin], s.banks[fout])
        s.banks[0].data.copy_(_to_bank(rows[0], nupts, neles))
        return dict(op='rhs', system=s)
    from frfs_amd.scattering import (DGFSBiScatteringModel, DGFSScatteringModel, subclass_where)
    from frfs_amd.velocitymesh import DGFSBiVelocityMesh, DGFSVelocityMesh
    cfg = _config(c)
    if c['model'] == 'vss':
        vm, base = DGFSBiVelocityMesh(be, cfg, c['species']), DGFSBiScatteringModel
    else:
        vm, base = DGFSVelocityMesh(be, cfg), DGFSScatteringModel
    model = subclass_where(base, scattering_model=cfg.get('scattering-model', 'type'))(be, cfg, vm)
    f = []
    for r in rows:
        m = be.matrix(shape)
        m.data.copy_(_to_bank(r, nupts, neles))
        f.append(m)
    q = [be.matrix(shape) for _ in range(c['species'])]
    state = dict(op=c['op'], model=model, f=f, q=q, bi=c['model'] == 'vss')
    if c['op'] == 'fs':
        state['elem'], state['upt'] = _where(c)
    return state


def _where(c):
    """The DOF of a per-DOF call."""
    return c['neles'] // 2, c['nupts'] - 1


def run(state):
    s = state
    if s['op'] == 'forward':
        s['net'].predict(s['g'], out=s['out'])
        return s['out']
    if s['op'] == 'gradient':
        sums, grad = s['net'].gradient(s['g'], s['t'])
        return {'sums': sums, 'grad': grad}
    if s['op'] == 'rhs':
        system = s['system']
        system.collide(0.0, 0, 1)
        system.rhs(0.0, 0, 2)
        system.axnpby(1, [1.0, (1.0, 2)])
        return {'rhs': system.banks[1].data, 'advection': system.banks[2].data}
    if s['op'] == 'fs':
        if s['bi']:
            s['model'].fs(s['elem'], s['upt'], *s['f'], *s['q'])
        else:
            s['model'].fs(*s['f'], *s['q'], s['elem'], s['upt'])
    else:
        s['model'].fs_batch(*s['f'], *s['q'])
    return [m.data for m in s['q']]


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    """Transforms are counted at 5 n log2 n: one complex transform for the two real-input items of a
    distinct product, half of one for each real product sum."""
    c = case
    n = c['Nv'] ** 3
    if c['op'] in ('forward', 'gradient'):
        lay, rows, modes = c['layers'], c['rows'], MODES ** 3
        point = 2 * WIDTH * WIDTH * n + 8 * WIDTH * n                     # channel matrix, activation
        spec = 2 * WIDTH * (2 * MODES * n + 4 * MODES ** 2 * n / c['Nv'] * 2) * 2 + 8 * WIDTH * WIDTH * modes
        weights = 4 * lay * (2 * WIDTH * WIDTH * modes + WIDTH * WIDTH)
        if c['op'] == 'forward':
            return {'bytes': 8 * n * rows + weights, 'flops': lay * rows * (point + spec)}
        return {'bytes': 8 * n * rows + 2 * weights, 'flops': 3 * lay * rows * (point + spec)}
    nupts, neles = _points(c)
    dofs = 1 if c['op'] == 'fs' else nupts * neles
    fft = 5 * n * math.log2(n)
    pairs = c['species'] * (c['species'] + 1) // 2
    if c['model'] == 'vss':
        prods = groups = c['Nrho'] * c['M'] // 2 * (pairs if c['species'] == 1 else 4)
    else:
        prods, groups = c['Nrho'] * c['M'] * (2 if c['model'] == 'nodal' else 1), c['Nrho']
    sources = 2 if c['model'] == 'nodal' else c['species']
    flops = dofs * (prods + 0.5 * groups + 0.5 * sources + c['species']) * fft
    moved = 8 * n * dofs * (sources + c['species'])
    if c['op'] == 'rhs':
        moved += 8 * n * dofs
        flops += dofs * n * (4 * (c['order'] + 1) + 16)
    return {'bytes': moved, 'flops': flops}


# ---------------------------------------------------------------- the same in 64 bits
def _design(npts):
    best = None
    for path in sorted(glob.glob(os.path.join(DESIGNS, 'womersley-*.txt'))):
        deg, m = (int(v) for v in re.search(r'-ss(\d+)-m(\d+)\.txt$', path).groups())
        if m == npts and (best is None or deg > best[0]):
            best = (deg, path)
    return np.loadtxt(best[1], ndmin=2)


def _radial(c):
    half = _dev(c)
    if c['model'] == 'vss':
        mr = max(_masses(c)) / ARGON['molarMass0']
        s = min(2 * half / (max(4 * mr / (1 + mr), 2) + math.sqrt(1 + mr) + 1),
                2 * half / (max(4 / (1 + mr), 2) + math.sqrt(1 + 1 / mr) + 1))
    else:
        s = 2 * half / (3 + math.sqrt(2))
    x, w = np.polynomial.legendre.leggauss(c['Nrho'])
    return s * (1 + x), s * w


def _freq(n):
    """Integer wave vectors (3, n, n, n), the unpaired index stored as -n/2."""
    k = torch.fft.fftfreq(n, 1.0 / n, dtype=torch.float64, device=_device())
    return torch.stack(torch.meshgrid(k, k, k, indexing='ij'))


def _inv(x):
    return torch.fft.ifftn(x, dim=(-3, -2, -1), norm='forward')


def _fwd(x):
    return torch.fft.fftn(x, dim=(-3, -2, -1))


def _sinc(x):
    return torch.sin(x + 1e-15) / (x + 1e-15)


def _number_density():
    return ARGON['rho0'] / ARGON['molarMass0'] * AVOGADRO


def _exact_vhs(c, f, g):
    """vhs-gll (g is f) and vhs-gll-nodal: Q(f, g) for (rows, n, n, n) inputs."""
    n, half = c['Nv'], _dev(c)
    qz, qw = _radial(c)
    sz, sw = _design(2 * c['M'])[:c['M']], 2 * math.pi / c['M']
    omega = 0.5
    gam = 2 * (1 - omega)
    inv_kn = ARGON['H0'] * math.sqrt(2) * math.pi * _number_density() * D_REF ** 2 * (T_REF / ARGON['T0']) ** (omega - 0.5)
    prefac = inv_kn / (2 ** (3 - omega) * math.gamma(2.5 - omega) * math.pi)
    l = _freq(n)
    size = l.square().sum(0).sqrt()
    ff = _fwd(f + 0j) / n ** 3
    fg = ff if g is f else _fwd(g + 0j) / n ** 3
    gain, bb2 = 0, 0
    for r in range(c['Nrho']):
        k = math.pi / half * qz[r]
        s = 0
        for q in range(c['M']):
            ph = torch.exp(0.5j * k * (sz[q, 0] * l[0] + sz[q, 1] * l[1] + sz[q, 2] * l[2]))
            if g is f:
                s = s + _inv(ph * ff) * _inv(ph.conj() * ff)
            else:
                s = s + 0.5 * (_inv(ph * ff) * _inv(ph.conj() * fg) + _inv(ph.conj() * ff) * _inv(ph * fg))
        gain = gain + (2 * qw[r] * sw / n ** 3) * qz[r] ** (gam + 2) * 4 * math.pi * _sinc(0.5 * k * size) * _fwd(s)
        bb2 = bb2 + qw[r] * qz[r] ** (gam + 2) * 16 * math.pi ** 2 * _sinc(k * size)
    return prefac * (_inv(gain).real - f * _inv(fg * bb2).real)


@functools.lru_cache(maxsize=2)
def _vss_tables(nv, nrho, m, species):
    """Gain weights b[pq][x][y] and loss weights c[pq]."""
    c = dict(Nv=nv, Nrho=nrho, M=m, species=species, model='vss')
    qz, qw = _radial(c)
    sz, pre = _design(m), _design(MPRE)
    mass = [v / ARGON['molarMass0'] for v in _masses(c)]
    l = _freq(nv)
    proj = torch.tensordot(torch.as_tensor(pre, device=l.device), l, dims=1)
    b, loss = {}, {}
    for pq, (alpha, omega, _, _) in _pairs(c).items():
        mq = mass[int(pq[1])] / (mass[int(pq[0])] + mass[int(pq[1])])
        wt = torch.as_tensor(np.maximum(1 + sz @ pre.T, 0) ** (alpha - 1), device=l.device) + 0j
        b[pq], loss[pq] = [], 0
        for x in range(nrho):
            k, scale = math.pi / _dev(c) * qz[x], 4 * math.pi / MPRE * qz[x] ** (2 * (1 - omega) + 2)
            b[pq].append(scale * torch.tensordot(wt, torch.exp(-1j * k * mq * proj), dims=1))
            loss[pq] = loss[pq] + qw[x] * 4 * math.pi / m * scale * torch.tensordot(wt.sum(0), torch.exp(-1j * k * proj), dims=1)
    return b, loss


def _exact_vss(c, fs):
    n, half, ns = c['Nv'], _dev(c), c['species']
    qz, qw = _radial(c)
    sz, sw = _design(c['M']), 4 * math.pi / c['M']
    mass = [v / ARGON['molarMass0'] for v in _masses(c)]
    b, loss = _vss_tables(n, c['Nrho'], c['M'], ns)
    l = _freq(n)
    ft = [_fwd(f + 0j) / n ** 3 for f in fs]
    out = []
    for p in range(ns):
        q_p = 0
        for q in range(ns):
            pq = '%d%d' % (p, q)
            alpha, omega, dref, tref = _pairs(c)[pq]
            kq, kp = mass[q] / (mass[p] + mass[q]), mass[p] / (mass[p] + mass[q])
            root, mu = math.sqrt(1 + mass[p] / mass[q]), mass[p] * mass[q] / (mass[p] + mass[q])
            inv_kn = root * math.pi * _number_density() * dref ** 2 * (tref / ARGON['T0']) ** (omega - 0.5) * ARGON['H0']
            prefac = inv_kn * alpha / (root * mu ** (omega - 0.5) * 2 ** (1 + alpha) * math.gamma(2.5 - omega) * math.pi)
            gain = 0
            for x in range(c['Nrho']):
                for y in range(c['M']):
                    a = math.pi / half * qz[x] * (sz[y, 0] * l[0] + sz[y, 1] * l[1] + sz[y, 2] * l[2])
                    s = _inv(torch.exp(1j * kq * a) * ft[p]) * _inv(torch.exp(-1j * kp * a) * ft[q])
                    gain = gain + (qw[x] * sw / n ** 3) * b[pq][x][y] * _fwd(s)
            q_p = q_p + prefac * (_inv(gain).real - fs[p] * _inv(loss[pq] * ft[q]).real)
        out.append(q_p)
    return out


def _project(c, qs):
    """Least-squares correction that zeroes each species' mass and the total momentum and energy."""
    n = c['Nv']
    cv = torch.as_tensor(_grid(n), dtype=torch.float64, device=qs[0].device)
    mass = [v / ARGON['molarMass0'] for v in _masses(c)] if c['model'] == 'vss' else [1.0]
    ns, pts = len(qs), n ** 3
    a = cv.new_zeros((ns + 4, ns, pts))
    for s in range(ns):
        a[s, s] = 1
        a[ns:ns + 3, s] = mass[s] * cv
        a[ns + 3, s] = mass[s] * cv.square().sum(0)
    a = a.reshape(ns + 4, -1)
    q = torch.stack([v.reshape(-1, pts) for v in qs], dim=1).reshape(-1, ns * pts)
    q = q - torch.linalg.solve(a @ a.T, a @ q.T).T @ a
    return [v.reshape(qs[0].shape) for v in q.reshape(-1, ns, pts).unbind(1)]


def _exact_collision(c, rows):
    n = c['Nv']
    step = max(1, int(256 * (32 / n) ** 3))
    parts = []
    for b in range(0, rows[0].shape[0], step):
        f = [r[b:b + step].reshape(-1, n, n, n) for r in rows]
        q = _exact_vss(c, f) if c['model'] == 'vss' else [_exact_vhs(c, f[0], f[-1] if c['model'] == 'nodal' else f[0])]
        q = _project(c, q) if c['project'] else q
        parts.append([v.reshape(-1, n ** 3) for v in q])
    return [torch.cat(p) for p in zip(*parts)]


def _exact_advection(c, f):
    """-div(c f): collocated derivatives on the Gauss points and the lifted jump to the upwind face flux."""
    p1, n = c['order'] + 1, c['Nv'] ** 3
    s = np.polynomial.legendre.leggauss(p1)[0]
    legendre = lambda x: np.stack([math.sqrt(k + 0.5) * np.polynomial.legendre.Legendre.basis(k)(x) for k in range(p1)])  # noqa: E731
    slope = np.stack([math.sqrt(k + 0.5) * np.polynomial.legendre.Legendre.basis(k).deriv()(s) for k in range(p1)])
    vinv = np.linalg.inv(legendre(s).T)
    diff, ends = slope.T @ vinv, legendre(np.array([-1.0, 1.0])).T @ vinv
    top = np.polynomial.legendre.Legendre.basis(p1 - 1)
    gx = np.concatenate([[-1.0], np.sort(top.deriv().roots().real) if p1 > 2 else [], [1.0]])
    gw = 2 / (p1 * (p1 - 1) * top(gx) ** 2)
    along = (legendre(s).T @ legendre(gx)) @ (gw[:, None] * (legendre(gx).T @ vinv))    # (point, face node)
    normal = legendre(s).T @ legendre(np.array([-1.0, 1.0]))                            # (point, end)
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=f.device)  # noqa: E731
    diff, ends, along, normal = t(diff), t(ends), t(along), t(normal)
    cv = t(_grid(c['Nv']))
    hx, hy = 1.0 / c['nelx'], 1.0 / c['nely']
    u = f.reshape(c['nely'], c['nelx'], p1, p1, n)
    out = torch.empty_like(u)
    for b in range(0, n, 2048):
        v = u[..., b:b + 2048]
        fx, fy = 0.5 * hy * cv[0, b:b + 2048], 0.5 * hx * cv[1, b:b + 2048]
        r = fx * torch.einsum('ij,yxajv->yxaiv', diff, v) + fy * torch.einsum('ij,yxjav->yxiav', diff, v)
        left, right = torch.einsum('ej,yxajv->eyxav', ends, v).unbind(0)
        low, high = torch.einsum('ej,yxjav->eyxav', ends, v).unbind(0)
        jump_r = fx * torch.where(fx > 0, torch.zeros_like(right), left.roll(-1, 1) - right)
        jump_l = -fx * torch.where(fx > 0, right.roll(1, 1) - left, torch.zeros_like(left))
        jump_h = fy * torch.where(fy > 0, torch.zeros_like(high), low.roll(-1, 0) - high)
        jump_l2 = -fy * torch.where(fy > 0, high.roll(1, 0) - low, torch.zeros_like(low))
        for jump, end in ((jump_l, 0), (jump_r, 1)):
            r = r + torch.einsum('i,ak,yxkv->yxaiv', normal[:, end], along, jump)
        for jump, end in ((jump_l2, 0), (jump_h, 1)):
            r = r + torch.einsum('i,ak,yxkv->yxiav', normal[:, end], along, jump)
        out[..., b:b + 2048] = -4 / (hx * hy) * r
    return out.reshape(-1, n)


def _network(c, theta, g):
    """The Fourier network on (rows, N^3) in 64 bits."""
    n, w, m = c['Nv'], WIDTH, MODES
    keep = torch.tensor(list(range(m // 2)) + list(range(n - m // 2, n)), device=g.device)
    at = 0

    def take(*shape):
        nonlocal at
        size = int(np.prod(shape))
        at += size
        return theta[at - size:at].reshape(shape)

    lift, bias = take(w), take(w)
    v = lift[:, None] * g[:, None] + bias[:, None]
    for layer in range(c['layers']):
        r, mat, off = torch.view_as_complex(take(w, w, m ** 3, 2)), take(w, w), take(w)
        x = torch.fft.fftn(v.reshape(-1, w, n, n, n), dim=(2, 3, 4), norm='forward')
        x = x[:, :, keep][:, :, :, keep][..., keep].reshape(-1, w, m ** 3)
        y = torch.matmul(x.permute(2, 0, 1), r.permute(2, 0, 1).contiguous()).permute(1, 2, 0).reshape(-1, w, m, m, m)
        full = torch.zeros((y.shape[0], w, n, n, n), dtype=y.dtype, device=y.device)
        i, j, k = torch.meshgrid(keep, keep, keep, indexing='ij')
        full = full.index_put((torch.arange(y.shape[0], device=y.device)[:, None, None, None, None],
                               torch.arange(w, device=y.device)[None, :, None, None, None], i, j, k), y)
        z = torch.matmul(mat, v) + off[:, None] + _inv(full).real.reshape(v.shape)
        v = torch.nn.functional.gelu(z) if layer < c['layers'] - 1 else z
    return (take(w)[:, None] * v).sum(1) + take(1)


def exact(case, seed):
    c = case
    if c['op'] in ('forward', 'gradient'):
        theta = torch.as_tensor(_theta(c['layers'], seed), device=_device()).double()
        g, t = _training_rows(c, seed)
        step = 32 if c['Nv'] == 16 else 4
        if c['op'] == 'forward':
            return torch.cat([_network(c, theta, g[b:b + step].double()) for b in range(0, c['rows'], step)])
        n = c['Nv'] ** 3
        count = c['rows'] * n
        cv = torch.as_tensor(_grid(c['Nv']), device=_device())
        phi = torch.stack([torch.ones_like(cv[0]), cv[0], cv[1], cv[2], cv.square().sum(0)])
        theta.requires_grad_(True)
        sums, grad = torch.zeros(3, dtype=torch.float64, device=theta.device), 0
        for b in range(0, c['rows'], step):
            out, tt = _network(c, theta, g[b:b + step].double()), t[b:b + step].double()
            u = torch.linalg.solve(phi @ phi.T, phi @ out.T).T @ phi
            e2, u2 = (out - tt).square().sum(), u.square().sum()
            grad = grad + torch.autograd.grad((e2 + 10.0 * u2) / count, theta)[0]
            sums += torch.stack([e2.detach(), tt.square().sum(), u2.detach()])
        return {'sums': sums, 'grad': grad}
    rows = _rows(c, seed)
    nupts, neles = _points(c)
    if c['op'] == 'fs':
        elem, upt = _where(c)
        d = elem * nupts + upt
        one = _exact_collision(c, [r[d:d + 1] for r in rows])
        out = []
        for q in one:
            full = torch.zeros((nupts * neles, q.shape[1]), dtype=torch.float64, device=q.device)
            full[d] = q[0]
            out.append(_to_bank(full, nupts, neles))
        return out
    q = _exact_collision(c, rows)
    if c['op'] == 'rhs':
        adv = _exact_advection(c, rows[0])
        return {'rhs': _to_bank(q[0] + adv, nupts, neles), 'advection': _to_bank(adv, nupts, neles)}
    return [_to_bank(v, nupts, neles) for v in q]
