"""The work that a user of this package has it do, as cases that can be timed
and compared: coupling matvecs and solves over lookup tables and over the
explicit matrix, and the fields computed from their solutions.

Geometry of every case: spheres (radius U(80, 120) nm, index U(1.5, 2.0) +
0.01i) in air above glass (n = 1.52), lambda = 550 nm, 2.78 spheres per um^2
with at least 20 nm between neighbours; one height for radial lookups, heights
U(150, 300) nm for volume lookups and the explicit matrix. exact() restates
the physics in torch at 64 bits without using the package.
"""
import math

import numpy as np
import torch

from smuthi_amd import cuda
from smuthi_amd.batch import EnsembleBatch
from smuthi_amd.expansions import PlaneWaveExpansion, SphericalWaveExpansion, SphericalWaveSum
from smuthi_amd.far_field import scattered_far_field
from smuthi_amd.layers import LayerSystem
from smuthi_amd.linear_system import CouplingMatrixExplicit, CouplingMatrixRadialLookupCUDA
from smuthi_amd.particles import Sphere
from smuthi_amd.volume import CouplingMatrixVolumeLookupCUDA

WL = 550.0
K = 2 * math.pi / WL
N_GLASS = 1.52
DENSITY = 2.78e-6  # spheres per nm^2
HEIGHT = 200.0     # nm, particles of the radial cases
Z_RANGE = (150.0, 300.0)
CLASSES = 24       # sphere kinds (radius, index) of one geometry


# ---- the cases -------------------------------------------------------------

def listed():
    return [
        # the 50 spheres on a substrate that also run on a CPU: one operator application, as any iterative
        # solver of the user's own asks for; latency is all there is
        dict(name='matvec_50', kind='matvec', n=50, l_max=3, h=5.0, neff=2e-3, interp='spline', precision='single',
             nrhs=1),
        # an FP64 application at a thousand spheres, the master matrix's LinearOperator; odd size, low order, linear
        dict(name='matvec_1023_fp64', kind='matvec', n=1023, l_max=2, h=5.5, neff=1e-2, interp='linear',
             precision='double', nrhs=1),
        # a block of right-hand sides at the higher order of the precision configuration
        dict(name='matvec_2501_block', kind='matvec', n=2501, l_max=4, h=5.0, neff=1e-2, interp='spline',
             precision='single', nrhs=8),
        # spheres at different heights: the two-table (volume) lookup, bicubic, a block that fills no batch
        dict(name='volume_700_block', kind='volume', n=701, l_max=3, h=8.0, neff=1e-2, interp='spline',
             precision='single', nrhs=3),
        # one incidence on a small ensemble: the default solve of a simulation
        dict(name='solve_50', kind='solve', n=50, l_max=3, h=5.0, neff=2e-3, interp='spline', precision='mixed',
             nrhs=1, tol=1e-6),
        # the headline: 10,000 spheres, eight incidences, 2 nm table, FP16-operand inner solves
        dict(name='solve_10000', kind='solve', n=10000, l_max=3, h=2.0, neff=2e-3, interp='spline',
             precision='mixed16', nrhs=8, tol=1e-6),
        # several ensembles and incidences in one batched solve over one volume table
        dict(name='ensembles_6x8', kind='ensembles', n=130, count=6, l_max=3, h=8.0, neff=1e-2, interp='catmull-rom',
             precision='mixed16', nrhs=8, tol=1e-6),
        # no lookup table: the explicit matrix of a small group of particles, built and solved by LU
        dict(name='explicit_lu_60', kind='explicit_lu', n=60, l_max=3, neff=1e-2, nrhs=1),
        # GMRES on a stored explicit matrix for an angular scan of incidences
        dict(name='explicit_gmres_300', kind='explicit_gmres', n=300, l_max=3, neff=1e-2, precision='mixed', nrhs=12,
             tol=1e-6),
        # the layer-mediated near field on a vertical cut above the particles
        dict(name='pwe_field_256', kind='pwe', nx=256, nz=256, n_kappa=1000, n_alpha=180, precision='single'),
        # the direct near field of a thousand spheres on the same kind of cut
        dict(name='swe_field_1000', kind='swe', n=1000, l_max=3, nx=192, nz=128, precision='single'),
        # the scattered far field on a one-degree grid (cross sections integrate it)
        dict(name='far_field_1000', kind='far', n=1000, l_max=3, step_deg=1.0, precision='double'),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(['matvec', 'matvec', 'matvec', 'volume', 'solve', 'solve', 'ensembles', 'explicit_lu',
                       'explicit_gmres', 'pwe', 'swe', 'far'])
    c = dict(kind=kind)
    if kind in ('matvec', 'volume'):
        l_max = rng.choice([1, 2, 3, 3, 4])
        # (a volume table of order 4 is large: two tables over heights and distances)
        c.update(n=log_int(20, 4000 if kind == 'matvec' else 300 if l_max == 4 else 800), l_max=l_max,
                 h=rng.choice([5.0, 5.5, 8.0]) if kind == 'matvec' else 8.0, neff=1e-2,
                 interp=rng.choice(['linear', 'spline', 'catmull-rom']))
        c['precision'], c['nrhs'] = rng.choice([('single', 1), ('double', 1), ('single', 8), ('single', 5),
                                                ('double', 8), ('half', 8), ('half', 11)])
    elif kind == 'solve':
        precision, nrhs = rng.choice([('mixed', 1), ('mixed', 8), ('double', 1), ('mixed16', 8), ('mixed16', 13)])
        c.update(n=log_int(20, 2000), l_max=rng.choice([2, 3]), h=5.0, neff=1e-2,
                 interp=rng.choice(['linear', 'spline']), precision=precision, nrhs=nrhs, tol=1e-6)
    elif kind == 'ensembles':
        c.update(n=log_int(20, 200), count=rng.randint(2, 8), l_max=3, h=8.0, neff=1e-2,
                 interp=rng.choice(['linear', 'catmull-rom']), precision=rng.choice(['mixed', 'mixed16']),
                 nrhs=rng.choice([1, 8]), tol=1e-6)
    elif kind == 'explicit_lu':
        c.update(n=log_int(5, 90), l_max=rng.choice([2, 3, 4]), neff=1e-2, nrhs=rng.choice([1, 3]))
    elif kind == 'explicit_gmres':
        c.update(n=log_int(20, 400), l_max=rng.choice([2, 3]), neff=1e-2, precision=rng.choice(['mixed', 'double']),
                 nrhs=rng.choice([1, 4, 12]), tol=1e-6)
    elif kind == 'pwe':
        c.update(nx=log_int(8, 300), nz=log_int(8, 250), n_kappa=log_int(150, 1500),
                 n_alpha=rng.choice([61, 120, 180, 361]), precision=rng.choice(['single', 'single', 'double']))
        if c['precision'] == 'double':
            c.update(nx=min(c['nx'], 130), nz=min(c['nz'], 100))
    elif kind == 'swe':
        c.update(n=log_int(20, 2000), l_max=rng.choice([2, 3, 4]), nx=log_int(16, 256), nz=log_int(16, 160),
                 precision=rng.choice(['single', 'single', 'double']))
    else:
        c.update(n=log_int(20, 2000), l_max=rng.choice([2, 3]), step_deg=rng.choice([1.0, 2.0, 3.0]),
                 precision=rng.choice(['single', 'double']))
    return c


# ---- inputs ------------------------------------------------------------------

def _seeded(case, seed):
    return np.random.default_rng([int(seed), case.get('n', 0), case.get('nx', 0), case.get('l_max', 0)])


def _geometry(n, rng, z_range=None):
    """(positions [n][3], class of each sphere, (radius, index) of the classes): a jittered square lattice,
    so that the density and the smallest gaps are those of a random monolayer."""
    a = 1 / math.sqrt(DENSITY)
    m = int(math.ceil(math.sqrt(n)))
    sites = rng.permutation(m * m)[:n]
    jitter = (a - 260.0) / 2  # two spheres of 120 nm radius and 20 nm between them
    xy = np.stack([sites % m, sites // m], axis=1) * a - m * a / 2 + rng.uniform(-jitter, jitter, (n, 2))
    z = np.full(n, HEIGHT) if z_range is None else rng.uniform(*z_range, n)
    kinds = [(float(r), complex(q, 0.01)) for r, q in zip(rng.uniform(80, 120, CLASSES), rng.uniform(1.5, 2.0, CLASSES))]
    return np.column_stack([xy, z]), rng.integers(0, CLASSES, n), kinds


def _contour(step):
    """k_parallel samples: along the real axis, below it past the branch points at 1 and 1.52, up to 2.7."""
    w = [0, 0.9, 0.9 - 0.01j, 1.72 - 0.01j, 1.72, 2.72]
    parts = []
    for a, b in zip(w[:-1], w[1:]):
        parts.append(a + (b - a) * np.linspace(0, 1, int(math.ceil(abs(b - a) / step)) + 1))
    return np.concatenate(parts).astype(complex) * K


def _spheres(pos, cls, kinds, l_max):
    return [Sphere(position=list(p), refractive_index=kinds[c][1], radius=kinds[c][0], l_max=l_max, m_max=l_max)
            for p, c in zip(pos, cls)]


def _incidences(rng, nrhs):
    """(polar angle, azimuth, polarisation) of plane waves from above."""
    return [(math.pi - math.radians(rng.uniform(0, 60)), rng.uniform(0, 2 * math.pi), j % 2) for j in range(nrhs)]


def _system_inputs(case, seed):
    """Positions, spheres' kinds, T-matrix diagonal and right-hand sides of a solve."""
    rng = _seeded(case, seed)
    radial = case['kind'] == 'solve'
    if case['kind'] == 'ensembles':
        sizes = [int(f) for f in np.linspace(0.6, 1.4, case['count']) * case['n']]  # uneven
    else:
        sizes = [case['n']]
    geo = [_geometry(s, rng, None if radial else Z_RANGE) for s in sizes]
    kinds = geo[0][2]
    pos = np.concatenate([g[0] for g in geo])
    cls = np.concatenate([g[1] for g in geo])
    t = _mie(kinds, case['l_max'])[cls]
    a = np.stack([_plane_wave(pos, case['l_max'], *inc) for inc in _incidences(rng, case['nrhs'])])
    rhs = (t[None] * a).reshape(case['nrhs'], -1)
    return sizes, pos, cls, kinds, t.reshape(-1), rhs


def _field_inputs(case, seed):
    rng = _seeded(case, seed)
    x, z = np.meshgrid(np.linspace(-10e3, 10e3, case['nx']) + rng.uniform(-5, 5),
                       np.linspace(330.0, 3000.0, case['nz']), indexing='ij')
    pts = np.stack([x.ravel(), np.full(x.size, rng.uniform(-50, 50)), z.ravel()], axis=1)
    return rng, pts


def _coefficients(rng, n, l_max):
    """Scattered-field coefficients: falling with l like a small sphere's."""
    _, l, _ = _orders(l_max)
    return (rng.standard_normal((n, len(l))) + 1j * rng.standard_normal((n, len(l)))) * 0.1 * 4.0 ** (1 - l)[None]


def _pwe_inputs(case, seed):
    rng, pts = _field_inputs(case, seed)
    kp = _contour(3.0 / case['n_kappa'])
    alpha = np.linspace(0, 2 * math.pi, case['n_alpha'])
    g = rng.standard_normal((2, len(kp), len(alpha))) + 1j * rng.standard_normal((2, len(kp), len(alpha)))
    # the reflected field of sources 200 nm above the substrate: evanescent waves have decayed on the way
    kz = _kz(kp, K)
    g *= np.exp(-np.abs(kz.imag) * 200.0)[None, :, None]
    return pts, kp, alpha, g


def _matvec_inputs(case, seed):
    rng = _seeded(case, seed)
    pos, cls, kinds = _geometry(case['n'], rng, None if case['kind'] == 'matvec' else Z_RANGE)
    n = case['n'] * _blocksize(case['l_max'])
    shape = (n,) if case['nrhs'] == 1 else (case['nrhs'], n)
    v = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    return pos, cls, kinds, v


def _interp(name):
    return dict(interpolator_kind='linear') if name == 'linear' else dict(interpolator_kind='cubic',
                                                                          cubic_interpolant=name)


def prepare(case, seed):
    cuda.enable_gpu()
    kind = case['kind']
    ls = LayerSystem([0, 0], [N_GLASS, 1])
    s = dict(case=case)
    if kind in ('matvec', 'volume'):
        pos, cls, kinds, s['v'] = _matvec_inputs(case, seed)
        make = CouplingMatrixRadialLookupCUDA if kind == 'matvec' else CouplingMatrixVolumeLookupCUDA
        s['op'] = make(WL, _spheres(pos, cls, kinds, case['l_max']), ls, k_parallel=_contour(case['neff']),
                       resolution=case['h'], **_interp(case['interp']))
    elif kind in ('solve', 'ensembles', 'explicit_lu', 'explicit_gmres'):
        sizes, pos, cls, kinds, s['t'], s['rhs'] = _system_inputs(case, seed)
        parts = _spheres(pos, cls, kinds, case['l_max'])
        kp = _contour(case['neff'])
        if kind == 'solve':
            s['op'] = CouplingMatrixRadialLookupCUDA(WL, parts, ls, k_parallel=kp, resolution=case['h'],
                                                     **_interp(case['interp']))
        elif kind == 'ensembles':
            off = np.concatenate([[0], np.cumsum(sizes)])
            s['op'] = EnsembleBatch(WL, [parts[a:b] for a, b in zip(off[:-1], off[1:])], ls, k_parallel=kp,
                                    resolution=case['h'], **_interp(case['interp'])).operator
        elif kind == 'explicit_gmres':
            s['op'] = CouplingMatrixExplicit(WL, parts, ls, k_parallel=kp)
        else:
            s.update(parts=parts, ls=ls, kp=kp)
    elif kind == 'pwe':
        pts, kp, alpha, g = _pwe_inputs(case, seed)
        s['pwe'] = PlaneWaveExpansion(K, kp, alpha, 'upgoing', [0, 0, 0], 0, np.inf)
        s['pwe'].coefficients = g
        s['pts'] = [np.ascontiguousarray(pts[:, c]) for c in range(3)]
    else:
        rng, pts = _field_inputs(case, seed) if kind == 'swe' else (_seeded(case, seed), None)
        pos, cls, kinds = _geometry(case['n'], rng)
        coef = _coefficients(rng, case['n'], case['l_max'])
        parts = _spheres(pos, cls, kinds, case['l_max'])
        for p, c in zip(parts, coef):
            p.scattered_field = SphericalWaveExpansion(K, p.l_max, p.m_max, 'outgoing', p.position, 0, np.inf)
            p.scattered_field.coefficients = c
        if kind == 'swe':
            s['field'] = SphericalWaveSum(K, parts, 0, np.inf)
            s['pts'] = [np.ascontiguousarray(pts[:, c]) for c in range(3)]
        else:
            step = math.radians(case['step_deg'])
            s.update(parts=parts, ls=ls, polar=np.arange(0, math.pi + step / 2, step),
                     azimuth=np.arange(0, 2 * math.pi + step / 2, step))
    return s


def run(s):
    case = s['case']
    kind = case['kind']
    if kind in ('matvec', 'volume'):
        return s['op'].matvec(s['v'], precision=case['precision'])
    if kind in ('solve', 'ensembles', 'explicit_gmres'):
        return s['op'].solve_master(s['t'], s['rhs'], case['tol'], precision=case['precision'])
    if kind == 'explicit_lu':
        op = CouplingMatrixExplicit(WL, s['parts'], s['ls'], k_parallel=s['kp'])
        return op.solve_master(s['t'], s['rhs'], 1e-6, precision='lu')
    if kind == 'pwe':
        return s['pwe'].electric_field(*s['pts'], precision=case['precision'])
    if kind == 'swe':
        return s['field'].electric_field(*s['pts'], precision=case['precision'])
    ff = scattered_far_field(WL, s['parts'], s['ls'], s['polar'], s['azimuth'], precision=case['precision'])
    return {'amplitude': ff.amplitude, 'signal': ff.signal}


# ---- what a pass cannot do without --------------------------------------------

def work(case):
    kind = case['kind']
    B = _blocksize(case.get('l_max', 1))
    taps = {'linear': 2, 'spline': 4, 'catmull-rom': 4}.get(case.get('interp'), 0)
    if kind in ('matvec', 'volume', 'solve', 'ensembles'):
        # every ordered pair's block interpolated once (4 flops per tap and entry) and applied (8 per right-hand
        # side); the table rows that a geometry of this extent spans and the vectors are read once
        n, R = case['n'], case['nrhs']
        pairs = case.get('count', 1) * n ** 2
        rho = math.sqrt(2 * n / DENSITY) / case['h']
        if kind in ('volume', 'ensembles'):
            nz = 2 * (Z_RANGE[1] - Z_RANGE[0]) / case['h'] + 6
            per, table = 4 * 2 * taps ** 2, 2 * min(rho * nz, pairs * taps ** 2)
        else:
            per, table = 4 * taps, min(rho, pairs * taps)
        size = 16 if case['precision'] == 'double' else 8
        vectors = 2 * case.get('count', 1) * n * B * R * 16
        steps = 1
        if kind in ('solve', 'ensembles'):
            steps = 10 if n > 300 else 7  # coupling products to 1e-6 at these sizes
        return dict(bytes=steps * (table * B * B * size + vectors), flops=steps * pairs * B * B * (per + 8 * R))
    if kind == 'explicit_lu':
        nk = len(_contour(case['neff']))
        n = case['n'] * B
        # the layer-mediated quadrature (two complex multiply-adds per kappa and entry) and the factorisation
        return dict(bytes=16.0 * n * n, flops=16.0 * nk * n * n + 8 / 3 * n ** 3)
    if kind == 'explicit_gmres':
        n = case['n'] * B
        size = 16 if case['precision'] == 'double' else 8
        return dict(bytes=7.0 * size * n * n, flops=7.0 * 8 * n * n * case['nrhs'])
    if kind == 'pwe':
        terms = float(case['nx'] * case['nz']) * len(_contour(3.0 / case['n_kappa'])) * case['n_alpha']
        return dict(bytes=case['nx'] * case['nz'] * 72 + 32 * terms / (case['nx'] * case['nz']), flops=36 * terms)
    if kind == 'swe':
        pairs = float(case['nx'] * case['nz']) * case['n']
        return dict(bytes=case['nx'] * case['nz'] * 72 + case['n'] * B * 16, flops=pairs * (19 * B + 150))
    dirs = (180 / case['step_deg']) * (360 / case['step_deg'])
    # top half: both directions of the particles' waves, bottom half: the downgoing one
    return dict(bytes=dirs * 48 + case['n'] * B * 16, flops=dirs * case['n'] * (8 * 3 * (2 * case['l_max'] + 1) + 20))


def tolerance(case):
    """About four times what the results were seen to differ from exact() by."""
    kind, precision = case['kind'], case.get('precision')
    if kind in ('matvec', 'volume'):
        return {'rel': {'single': 3e-6, 'double': 1e-13, 'half': 2e-3}[precision]}
    if kind in ('solve', 'ensembles', 'explicit_gmres'):
        return {'rel': 5e-6}  # two solutions that each meet the 1e-6 residual
    if kind == 'explicit_lu':
        return {'rel': 1e-12}
    if precision == 'double':
        return {'rel': 1e-12}
    return {'rel': 1e-5 if kind == 'far' else 6e-6}


# ---- 64-bit reference ----------------------------------------------------------

def _blocksize(l_max):
    return 2 * l_max * (l_max + 2)


def _orders(l_max):
    """(tau, l, m) over the multipole index."""
    q = [(t, l, m) for t in range(2) for l in range(1, l_max + 1) for m in range(-l, l + 1)]
    return tuple(np.array(v) for v in zip(*q))


def _kz(kappa, k):
    kz = np.sqrt(k ** 2 - np.asarray(kappa) ** 2 + 0j)
    return np.where(kz.imag < 0, -kz, kz)


def _legendre(ct, st, l_max):
    """Normalised P, pi, tau [l][m] (integral of P^2 over cos theta = 1) as dicts; any array type."""
    P, pi, tau = {}, {}, {}
    one = ct * 0 + 1
    for m in range(l_max + 1):
        c = math.sqrt(0.5)
        for t in range(1, m + 1):
            c *= math.sqrt((2 * t + 1) / (2 * t))
        lo = max(m, 1)
        # p = P / st for m >= 1 (that is pi), P itself for m = 0
        p = {m: one * c * (st ** (m - 1) if m else 1), m - 1: one * 0}
        for l in range(m, l_max):
            a = math.sqrt((2 * l + 1) * (2 * l + 3) / ((l + 1 - m) * (l + 1 + m)))
            b = math.sqrt((2 * l + 3) * (l - m) * (l + m) / ((2 * l - 1) * (l + 1 - m) * (l + 1 + m))) if l > m else 0
            p[l + 1] = a * ct * p[l] - b * p[l - 1]
        for l in range(m, l_max + 1):
            P[l, m] = p[l] * (st if m else 1)
            pi[l, m] = p[l] if m else one * 0
        for l in range(lo, l_max + 1):
            if m:
                e = math.sqrt((2 * l + 1) * (l - m) * (l + m) / (2 * l - 1))
                tau[l, m] = l * ct * p[l] - e * p[l - 1]
    for l in range(1, l_max + 1):  # dP_l^0/dtheta = -sqrt(l (l + 1)) P_l^1
        tau[l, 0] = -math.sqrt(l * (l + 1)) * P[l, 1]
    return P, pi, tau


def _b_coefficients(l_max, ct, st, dagger):
    """Plane-wave / spherical-wave conversion coefficients [pol][n] (numpy arrays over ct)."""
    _, pi, tau = _legendre(ct, st, l_max)
    u = -1j if dagger else 1j
    out = [[], []]
    for t, l, m in zip(*_orders(l_max)):
        for pol in range(2):
            f = tau[l, abs(m)] if t == pol else m * pi[l, abs(m)]
            out[pol].append(-1 / u ** (l + 1) / math.sqrt(2 * l * (l + 1)) * (u if pol == 0 else 1) * f)
    return np.array(out)


def _fresnel(kappa):
    """(reflection, transmission) [pol] for waves falling from air on the glass."""
    ka, kg, n2 = _kz(kappa, K), _kz(kappa, K * N_GLASS), N_GLASS ** 2
    r = [(ka - kg) / (ka + kg), (n2 * ka - kg) / (n2 * ka + kg)]
    t = [2 * ka / (ka + kg), 2 * N_GLASS * ka / (n2 * ka + kg)]
    return np.array(r), np.array(t)


def _plane_wave(pos, l_max, polar, azimuth, pol):
    """Regular coefficients [particle][n] of a plane wave from above and its reflection."""
    kp, kz = K * math.sin(polar), K * math.cos(polar)  # kz < 0
    _, _, m = _orders(l_max)
    r, _ = _fresnel(np.array([kp]))
    phase = np.exp(1j * kp * (pos[:, 0] * math.cos(azimuth) + pos[:, 1] * math.sin(azimuth)))
    out = 0
    for s, amp in ((kz, 1.0), (-kz, r[pol, 0])):
        b = _b_coefficients(l_max, np.array([s / K]), np.array([kp / K]), True)[pol, :, 0]
        out = out + 4 * amp * (phase * np.exp(1j * s * pos[:, 2]))[:, None] * (b * np.exp(-1j * m * azimuth))[None]
    return out


def _riccati(l_max, z):
    """x j_l(x), x h_l(x) and their derivatives for l = 1..l_max at one complex argument."""
    top = l_max + 30
    j = [0j] * (top + 2)
    j[top] = 1e-30
    for l in range(top, 0, -1):
        j[l - 1] = (2 * l + 1) / z * j[l] - j[l + 1]
    scale = np.sin(z) / z / j[0]
    j = [v * scale for v in j]
    h = [-1j * np.exp(1j * z) / z, -np.exp(1j * z) * (z + 1j) / z ** 2]
    for l in range(1, l_max + 1):
        h.append((2 * l + 1) / z * h[l] - h[l - 1])
    return [(j[l], z * j[l - 1] - l * j[l], h[l], z * h[l - 1] - l * h[l]) for l in range(1, l_max + 1)]


def _mie(kinds, l_max):
    """Diagonal of the T-matrix of each sphere kind in air."""
    tau, l, _ = _orders(l_max)
    out = []
    for radius, n in kinds:
        q = {}
        for i, (a, b) in enumerate(zip(_riccati(l_max, complex(K * radius)), _riccati(l_max, n * K * radius))):
            (jm, djm, hm, dhm), (jp, djp, _, _) = a, b
            q[0, i + 1] = (jm * djp - jp * djm) / (jp * dhm - hm * djp)
            q[1, i + 1] = (jm * djp - n ** 2 * jp * djm) / (n ** 2 * jp * dhm - hm * djp)
        out.append([q[t, i] for t, i in zip(tau, l)])
    return np.array(out)


def _three_j(l1, l2, l3, m1, m2, m3):
    if m1 + m2 + m3 or not abs(l1 - l2) <= l3 <= l1 + l2 or abs(m3) > l3:
        return 0.0
    f = math.factorial
    pre = (f(l1 + l2 - l3) * f(l1 - l2 + l3) * f(l2 + l3 - l1) / f(l1 + l2 + l3 + 1)
           * f(l1 + m1) * f(l1 - m1) * f(l2 + m2) * f(l2 - m2) * f(l3 + m3) * f(l3 - m3))
    s = 0.0
    for k in range(l1 + l2 + l3 + 1):
        d = (k, l1 + l2 - l3 - k, l1 - m1 - k, l2 + m2 - k, l3 - l2 + m1 + k, l3 - l1 - m2 + k)
        if min(d) >= 0:
            s += (-1.0) ** k / math.prod(f(v) for v in d)
    return (-1.0) ** (l1 - l2 - m3) * s * math.sqrt(pre)


def _translation(l_max):
    """c[n1, n2, p]: outgoing wave n2 seen as regular waves n1, sum_p c h_p(kd) P_p^|m1-m2|(cos) e^{i(m2-m1)phi}."""
    q = [tuple(int(v) for v in n) for n in zip(*_orders(l_max))]
    c = np.zeros((len(q), len(q), 2 * l_max + 1), complex)
    for i, (t1, l2, m2) in enumerate(q):
        for j, (t2, l1, m1) in enumerate(q):
            for p in range(max(abs(l1 - l2), abs(m1 - m2)), l1 + l2 + 1):
                u = 1j ** (abs(m1 - m2) - abs(m1) - abs(m2) + l2 - l1 + p) * (-1.0) ** (m1 - m2)
                u *= math.sqrt((2 * l1 + 1) * (2 * l2 + 1) * (2 * p + 1) / (2 * l1 * (l1 + 1) * l2 * (l2 + 1)))
                w = _three_j(l1, l2, p, m1, -m2, m2 - m1)
                if t1 == t2:
                    w *= (l1 * (l1 + 1) + l2 * (l2 + 1) - p * (p + 1)) * _three_j(l1, l2, p, 0, 0, 0)
                elif p:
                    w *= math.sqrt((l1 + l2 + 1 + p) * (l1 + l2 + 1 - p) * (p + l1 - l2) * (p - l1 + l2))
                    w *= _three_j(l1, l2, p - 1, 0, 0, 0)
                else:
                    w = 0.0
                c[i, j, p] = u * w
    return c


def _device():
    return torch.device('cuda' if torch.cuda.is_available() else 'cpu')


def _tensor(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(_device())


def _hankel(n_max, x):
    """Spherical h_0..h_n_max of a real tensor x > 0."""
    e = torch.exp(1j * x)
    h = [-1j * e / x, -e * (x + 1j) / x ** 2]
    for l in range(1, n_max):
        h.append((2 * l + 1) / x * h[l] - h[l - 1])
    return h[:n_max + 1]


def _bessel(n_max, z):
    """J_0..J_n_max [n, ...] of a complex tensor: the integral over one period by the trapezoid rule for
    |z| < 40, Hankel's asymptotic expansion beyond."""
    out = torch.zeros((n_max + 1,) + z.shape, dtype=torch.complex128, device=z.device)
    far = (z.abs() >= 40) & (z.real > 0)
    near, big = z[~far], z[far]
    theta = torch.arange(120, dtype=torch.float64, device=z.device) * (2 * math.pi / 120)
    e = torch.exp(1j * near[:, None] * torch.sin(theta)[None])
    for n in range(n_max + 1):
        out[n][~far] = e @ torch.exp(-1j * n * theta) / 120
        mu, term, p, q = 4.0 * n * n, torch.ones_like(big), torch.ones_like(big), torch.zeros_like(big)
        for k in range(1, 31):
            term = term * (mu - (2 * k - 1) ** 2) / (k * 8 * big)
            s = 1 if k % 4 < 2 else -1
            if k % 2:
                q = q + s * term
            else:
                p = p + s * term
        chi = big - (n / 2 + 0.25) * math.pi
        out[n][far] = torch.sqrt(2 / (math.pi * big)) * (torch.cos(chi) * p - torch.sin(chi) * q)
    return out


def _direct(l_max, rho, dz):
    """Direct coupling [..., B, B] without the azimuthal phase at real tensors rho, dz."""
    d = torch.sqrt(rho ** 2 + dz ** 2)
    P, _, _ = _legendre(dz / d, rho / d, 2 * l_max)
    h = _hankel(2 * l_max, K * d)
    c = _tensor(_translation(l_max))
    _, _, m = _orders(l_max)
    dm = np.abs(m[:, None] - m[None])
    out = torch.zeros(rho.shape + c.shape[:2], dtype=torch.complex128, device=rho.device)
    for q in range(2 * l_max + 1):
        i, j = (_tensor(v) for v in np.nonzero(dm == q))
        f = torch.stack([h[p] * P[p, q] for p in range(q, 2 * l_max + 1)], dim=-1)
        out[..., i, j] = f @ c[i, j, q:].T
    return out


def _reflected(l_max, kappa, rho, sz, drop_last):
    """Coupling through the substrate [..., B, B] without the azimuthal phase at z1 + z2 = sz."""
    kz = _kz(kappa, K)
    w = np.zeros(len(kappa), complex)
    d = np.diff(kappa)[:-1] if drop_last else np.diff(kappa)
    w[:len(d)] += d
    w[1:len(d) + 1] += d
    r, _ = _fresnel(kappa)
    bd = _b_coefficients(l_max, kz / K, kappa / K, True)
    bn = _b_coefficients(l_max, -kz / K, kappa / K, False)
    _, _, m = _orders(l_max)
    dm = np.abs(m[:, None] - m[None])
    pre = (2 * w * kappa / (kz * K))
    coef = np.einsum('pk,pik,pjk->kij', r * pre[None], bd, bn) * (1j ** dm)[None]
    coef, shape = _tensor(coef), rho.shape
    rho, sz = rho.reshape(-1), torch.broadcast_to(sz, rho.shape).reshape(-1)
    out = torch.zeros((len(rho),) + dm.shape, dtype=torch.complex128, device=rho.device)
    kt, kzt = _tensor(kappa), _tensor(kz)
    for a in range(0, len(rho), 4096):
        s = slice(a, a + 4096)
        J = _bessel(2 * l_max, rho[s, None] * kt[None])
        e = torch.exp(1j * kzt[None] * sz[s, None])
        for q in range(2 * l_max + 1):
            i, j = (_tensor(v) for v in np.nonzero(dm == q))
            out[s][:, i, j] = (J[q] * e) @ coef[:, i, j]
    return out.reshape(shape + dm.shape)


def _moments(y, dim):
    """h^2 / 6 times the second derivatives of the not-a-knot cubic splines through y along one axis."""
    y = y.movedim(dim, 0)
    n = y.shape[0]
    rhs = y[:-2] - 2 * y[1:-1] + y[2:]
    m = torch.zeros_like(y)
    m[1], m[n - 2] = rhs[0] / 6, rhs[n - 3] / 6
    c, d = {}, {}
    for j in range(2, n - 2):
        v = rhs[j - 1]
        v = v - m[1] if j == 2 else v - d[j - 1]
        if j == n - 3:
            v = v - m[n - 2]
        den = 4.0 - (c[j - 1] if j > 2 else 0.0)
        c[j], d[j] = 1 / den, v / den
    for j in range(n - 3, 1, -1):
        m[j] = d[j] - (c[j] * m[j + 1] if j < n - 3 else 0)
    m[0], m[n - 1] = 2 * m[1] - m[2], 2 * m[n - 2] - m[n - 3]
    return m.movedim(0, dim)


def _taps(interp, w):
    """[(moment?, row offset, weight)] of the interpolant at bin fraction w."""
    v = 1 - w
    if interp == 'linear':
        return [(0, 0, v), (0, 1, w)]
    if interp == 'spline':
        return [(0, 0, v), (0, 1, w), (1, 0, v ** 3 - v), (1, 1, w ** 3 - w)]
    return [(0, -1, -0.5 * w * v * v), (0, 0, 1 - 2.5 * w ** 2 + 1.5 * w ** 3),
            (0, 1, 0.5 * w + 2 * w ** 2 - 1.5 * w ** 3), (0, 2, -0.5 * w * w * v)]


def _rounded(t):
    return t.to(torch.complex64).to(torch.complex128)


def _lookup(case, sizes, pos, kappa):
    """A function of receiver and emitter indices to the coupling blocks [pairs, B, B] that the lookup of this
    case interpolates, azimuthal phases included."""
    h, l_max = case['h'], case['l_max']
    xyz = _tensor(pos)
    off = np.concatenate([[0], np.cumsum(sizes)])
    rho_max, rho_min = 0.0, math.inf
    for a, b in zip(off[:-1], off[1:]):
        d = torch.cdist(xyz[a:b, :2], xyz[a:b, :2], compute_mode='donot_use_mm_for_euclid_dist')
        rho_max = max(rho_max, float(d.max()))
        d.fill_diagonal_(math.inf)
        rho_min = min(rho_min, float(d.min()))
    rho = _tensor(np.arange(-3 * h, rho_max + 3 * h, h))
    shown = rho >= rho_min / 2
    _, _, m = _orders(l_max)
    mdiff = _tensor((m[None] - m[:, None]).astype(float))
    radial = case['kind'] in ('matvec', 'solve')
    if radial:
        sz = torch.full_like(rho, 2 * HEIGHT)
        direct = torch.zeros(rho.shape + mdiff.shape, dtype=torch.complex128, device=rho.device)
        direct[shown] = _direct(l_max, rho[shown], torch.zeros_like(rho[shown]))
        tabs = [(_rounded(direct) + _reflected(l_max, kappa, rho, sz, False), None)]
    else:
        z0, z1 = float(pos[:, 2].min()), float(pos[:, 2].max())
        sz = _tensor(np.arange(2 * z0 - 3 * h, 2 * z1 + 3 * h, h))
        dz = _tensor(np.arange(z0 - z1 - 3 * h, z1 - z0 + 3 * h, h))
        direct = torch.zeros((len(rho), len(dz)) + mdiff.shape, dtype=torch.complex128, device=rho.device)
        R, Z = torch.meshgrid(rho[shown], dz, indexing='ij')
        direct[shown] = _direct(l_max, R, Z)
        R, Z = torch.meshgrid(rho, sz, indexing='ij')
        tabs = [(_rounded(_reflected(l_max, kappa, R, Z, False)), (1, float(sz[0]))),
                (_rounded(direct), (-1, float(dz[0])))]
    cubic = case['interp'] == 'spline'
    full = []
    for t, axis in tabs:  # [moment along rho][moment along z]
        mr = _moments(t, 0) if cubic else None
        rows = [[t, _moments(t, 1) if cubic and axis else None], [mr, _moments(mr, 1) if cubic and axis else None]]
        full.append((rows, axis))

    def blocks(i, j):
        d = xyz[i] - xyz[j]
        r = torch.sqrt(d[:, 0] ** 2 + d[:, 1] ** 2)
        u = (r - rho[0]) / h
        a = torch.floor(u)
        phi = torch.atan2(d[:, 1], d[:, 0])
        out = 0
        for rows, axis in full:
            zt = [(0, 0, None)]
            if axis:
                uz = (xyz[i, 2] + axis[0] * xyz[j, 2] - axis[1]) / h
                b = torch.floor(uz)
                zt = _taps(case['interp'], uz - b)
            for mr, dr, wr in _taps(case['interp'], u - a):
                for mz, dzo, wz in zt:
                    t = rows[mr][mz]
                    row = t[a.long() + dr] if wz is None else t[a.long() + dr, b.long() + dzo]
                    out = out + (wr if wz is None else wr * wz)[:, None, None] * row
        return out * torch.exp(1j * phi[:, None, None] * mdiff[None])

    return blocks


def _explicit(case, pos, kappa):
    """The explicit coupling matrix [n B, n B]: every pair at its own distance and heights."""
    l_max, n = case['l_max'], len(pos)
    xyz = _tensor(pos)
    _, _, m = _orders(l_max)
    mdiff = _tensor((m[None] - m[:, None]).astype(float))
    B = len(m)
    W = torch.zeros((n, B, n, B), dtype=torch.complex128, device=xyz.device)
    for i in range(n):
        d = xyz[i][None] - xyz
        rho = torch.sqrt(d[:, 0] ** 2 + d[:, 1] ** 2)
        blk = _reflected(l_max, kappa, rho, xyz[i, 2] + xyz[:, 2], True)
        o = torch.arange(n, device=xyz.device) != i
        blk[o] += _direct(l_max, rho[o], d[o, 2])
        blk = blk * torch.exp(1j * torch.atan2(d[:, 1], d[:, 0])[:, None, None] * mdiff[None])
        W[i] = blk.permute(1, 0, 2)
    return W.reshape(n * B, n * B)


def _exact_matvec(case, seed):
    pos, _, _, v = _matvec_inputs(case, seed)
    n, B = case['n'], _blocksize(case['l_max'])
    blocks = _lookup(case, [n], pos, _contour(case['neff']))
    x = _tensor(v).reshape(case['nrhs'], n, B).permute(1, 2, 0).contiguous()
    y = torch.zeros_like(x)
    step = max(1, int(2e7 / (n * B * B)))
    idx = torch.arange(n, device=x.device)
    for a in range(0, n, step):
        r = idx[a:a + step]
        L = blocks(r.repeat_interleave(n), idx.repeat(len(r)))
        y[a:a + step] = torch.matmul(L.reshape(len(r), n, B, B), x[None]).sum(1)
    return y.permute(2, 0, 1).reshape(v.shape).cpu().numpy()


def _exact_solve(case, seed):
    sizes, pos, _, _, t, rhs = _system_inputs(case, seed)
    B, kappa = _blocksize(case['l_max']), _contour(case['neff'])
    t, rhs = _tensor(t), _tensor(rhs)
    x = torch.zeros_like(rhs)
    blocks = _explicit(case, pos, kappa) if 'interp' not in case else _lookup(case, sizes, pos, kappa)
    a = 0
    for n in sizes:
        if 'interp' in case:
            idx = torch.arange(a, a + n, device=t.device)
            W = torch.cat([blocks(i.repeat(n), idx).permute(1, 0, 2).reshape(B, n * B) for i in idx])
        else:
            W = blocks
        s = slice(a * B, (a + n) * B)
        M = torch.eye(n * B, dtype=W.dtype, device=W.device) - t[s, None] * W
        x[:, s] = torch.linalg.solve(M, rhs[:, s].T).T
        a += n
    return x.cpu().numpy()


def _exact_pwe(case, seed):
    pts, kp, alpha, g = _pwe_inputs(case, seed)
    kz = _kz(kp, K)
    dk, da = np.diff(kp), np.diff(alpha)
    wk, wa = np.zeros(len(kp), complex), np.zeros(len(alpha))
    wk[:-1], wa[:-1] = dk / 2, da / 2
    wk[1:] += dk / 2
    wa[1:] += da / 2
    c, s, q = np.cos(alpha)[None], np.sin(alpha)[None], (kz / K)[:, None]
    f = np.stack([-s * g[0] + c * q * g[1], c * g[0] + s * q * g[1], -(kp / K)[:, None] * g[1]])
    f = _tensor(f * (wk * kp)[None, :, None] * wa[None, None])
    p, kpt, kzt, ct, st = _tensor(pts), _tensor(kp), _tensor(kz), _tensor(np.cos(alpha)), _tensor(np.sin(alpha))
    out = torch.zeros((3, len(pts)), dtype=torch.complex128, device=p.device)
    u = p[:, 0, None] * ct[None] + p[:, 1, None] * st[None]
    for k in range(len(kp)):
        e = torch.exp(1j * (kpt[k] * u + kzt[k] * p[:, 2, None]))
        out += (e @ f[:, k].T).T
    return tuple(out.cpu().numpy())


def _exact_swe(case, seed):
    rng, pts = _field_inputs(case, seed)
    pos, cls, kinds = _geometry(case['n'], rng)
    coef = _tensor(_coefficients(rng, case['n'], case['l_max']))
    p, radius = _tensor(pts), [kinds[c][0] for c in cls]
    out = torch.zeros((3, len(pts)), dtype=torch.complex128, device=p.device)
    for i in range(case['n']):
        d = p - _tensor(pos[i])[None]
        r = torch.sqrt((d ** 2).sum(1))
        rho = torch.sqrt(d[:, 0] ** 2 + d[:, 1] ** 2)
        ct, st = d[:, 2] / r, rho / r
        cp, sp = torch.where(rho > 0, d[:, 0] / rho, 1.0), torch.where(rho > 0, d[:, 1] / rho, 0.0)
        P, pi, tau = _legendre(ct, st, case['l_max'])
        h = _hankel(case['l_max'], K * r)
        er, et, ep = 0, 0, 0  # spherical components
        for n, (t, l, m) in enumerate(zip(*_orders(case['l_max']))):
            l, m = int(l), int(m)
            a = coef[i, n] * (cp + 1j * sp) ** m / math.sqrt(2 * l * (l + 1))
            if t == 0:
                et, ep = et + a * h[l] * 1j * m * pi[l, abs(m)], ep - a * h[l] * tau[l, abs(m)]
            else:
                g = h[l - 1] - l * h[l] / (K * r)
                er = er + a * l * (l + 1) * h[l] / (K * r) * P[l, abs(m)]
                et, ep = et + a * g * tau[l, abs(m)], ep + a * g * 1j * m * pi[l, abs(m)]
        f = torch.stack([er * st * cp + et * ct * cp - ep * sp, er * st * sp + et * ct * sp + ep * cp,
                         er * ct - et * st])
        out += f * (r > radius[i])[None]
    return tuple(out.cpu().numpy())


def _exact_far(case, seed):
    rng = _seeded(case, seed)
    pos, _, _ = _geometry(case['n'], rng)
    coef, p = _tensor(_coefficients(rng, case['n'], case['l_max'])), _tensor(pos)
    step = math.radians(case['step_deg'])
    polar, az = np.arange(0, math.pi + step / 2, step), _tensor(np.arange(0, 2 * math.pi + step / 2, step))
    _, _, m = _orders(case['l_max'])
    em = torch.exp(1j * _tensor(m.astype(float))[:, None] * az[None])  # [n, alpha]
    amp, sig = [], []
    for top, beta in ((True, polar[polar < math.pi / 2]), (False, polar[polar > math.pi / 2])):
        n0 = 1.0 if top else N_GLASS
        for b in beta:
            kp = np.array([K * n0 * math.sin(b)])
            ka, kl = _kz(kp, K)[0], _kz(kp, K * n0)[0]
            r, t = _fresnel(kp)
            ph = torch.exp(-1j * float(kp[0]) * (p[:, 0, None] * torch.cos(az) + p[:, 1, None] * torch.sin(az)))
            g = []
            for s in (1, -1):
                bt = _tensor(_b_coefficients(case['l_max'], np.array([s * ka / K]), kp / K + 0j, False)[:, :, 0]
                             / (2 * math.pi * ka * K))
                c = coef * torch.exp(-1j * s * complex(ka) * p[:, 2, None])
                d = c.T.to(ph.dtype) @ ph  # [n, alpha]
                g.append(torch.stack([(bt[q][:, None] * em * d).sum(0) for q in range(2)]).cpu().numpy())
            g = g[0] + r * g[1] if top else t * g[1]
            amp.append(-2 * math.pi * kl * K * n0 * g)
            sig.append((2 * math.pi ** 2 / K * kl ** 2 * K * n0 * np.abs(g) ** 2).real)
    return {'amplitude': np.stack(amp, axis=1), 'signal': np.stack(sig, axis=1)}


def exact(case, seed):
    kind = case['kind']
    if kind in ('matvec', 'volume'):
        return _exact_matvec(case, seed)
    if kind in ('solve', 'ensembles', 'explicit_lu', 'explicit_gmres'):
        # a dense solve of all unknowns
        return _exact_solve(case, seed) if case['n'] <= 400 else None
    return {'pwe': _exact_pwe, 'swe': _exact_swe, 'far': _exact_far}[kind](case, seed)
