"""PWE fields of compact leaves (azimuthal harmonics with Bessel functions) and of
wide ones (one term per azimuth), over what decides between them and sizes
their work: points above one another (order 0), dense patches that need a few,
up to 31 and up to 63 orders, leaves that mix points on and off their axis,
azimuths below, at and beyond a staging chunk of 192 and too few for the
harmonics, kappa counts that fill no group of eight, real and lossy contours,
E and H, up- and downgoing, one discrete wave. Reference: the oracle's nested
trapezoid sums. Bounds, relative to the largest field: FP64 keeps 1e-16 per
term and truncates at 1e-16, 1e-10 as the kernel's own test; FP32 rounds
coefficients, azimuth sums and phases (6e-8 of numbers up to |k| times the
leaf's extent), 5e-5 as that test where leaves are wide and 3e-6 where they are
compact."""
import numpy as np
import pytest

from oracle import system as osys

pytestmark = pytest.mark.gpu

WL = 550.0
K = 2 * np.pi / WL


@pytest.fixture(scope='module')
def gpu():
    from smuthi_amd import cuda
    assert cuda.enable_gpu(), 'MI355X not available'
    return cuda


def _points(shape, rng):
    if shape == 'grid':       # a vertical cut: columns of 20 points, and ten points of a column of their own
        x, z = np.meshgrid(np.linspace(-900, 900, 31), np.linspace(20, 700, 20))
        p = np.stack([x.ravel(), np.full(x.size, 15.0), z.ravel()], 1)
        return np.concatenate([p, np.stack([np.zeros(10), np.zeros(10), np.linspace(50, 60, 10)], 1)])
    if shape == 'columns':    # two columns of 300 points and one point beside them
        z = np.linspace(20, 900, 300)
        p = [np.stack([np.full(300, x), np.full(300, 40.0), z], 1) for x in (-700.0, 650.0)]
        return np.concatenate(p + [np.array([[0.0, 0.0, 50.0]])])
    if shape == 'line':       # along x, the leaf's centre among the points
        return np.stack([np.linspace(-800, 800, 513), np.zeros(513), np.full(513, 100.0)], 1)
    if shape == 'volume':     # every leaf tall, points at random
        return np.stack([rng.uniform(-300, 300, 700), rng.uniform(-300, 300, 700), rng.uniform(20, 600, 700)], 1)
    if shape == 'one':
        return np.array([[123.0, -45.0, 67.0]])
    r = {'patch': 250.0, 'wide patch': 700.0, 'sparse': 4000.0}[shape]
    return np.stack([rng.uniform(-r, r, 255), rng.uniform(-r, r, 255), rng.uniform(20, 120, 255)], 1)


@pytest.mark.parametrize('n_k,n_a,neff,lossy', [(9, 64, 1.6, True), (30, 193, 2.7, True), (17, 385, 1.6, False),
                                                (8, 5, 1.6, True), (1, 1, 0.6, False)])
@pytest.mark.parametrize('shape', ['columns', 'grid', 'line', 'volume', 'one', 'patch', 'wide patch', 'sparse'])
def test_fields_match_oracle(gpu, shape, n_k, n_a, neff, lossy):
    from smuthi_amd.expansions import PlaneWaveExpansion
    rng = np.random.default_rng(n_k + n_a)
    pts = _points(shape, rng)
    kp = (np.linspace(0.0, neff, n_k) if n_k > 1 else np.array([neff])) * K + 0j
    if lossy:
        kp[n_k // 3:2 * n_k // 3] -= 0.01j * K
    alpha = np.linspace(0, 2 * np.pi, n_a) if n_a > 1 else np.array([0.7])
    g = rng.standard_normal((2, n_k, n_a)) + 1j * rng.standard_normal((2, n_k, n_a))
    kind = 'downgoing' if n_k == 17 else 'upgoing'
    x, y, z = pts.T * (np.array([1, 1, -1])[:, None] if kind == 'downgoing' else 1)
    made = []
    for cls in (osys.PlaneWaveExpansion, PlaneWaveExpansion):
        e = cls(K, kp, alpha, kind, [30.0, -20.0, 0.0], -np.inf, np.inf)
        e.coefficients = g.copy()
        made.append(e)
    print('pwe harmonics: %s, %d x %d waves' % (shape, n_k, n_a), flush=True)
    for field in ('electric_field', 'magnetic_field'):
        args = (x, y, z) if field == 'electric_field' else (x, y, z, WL)
        want = np.stack(getattr(made[0], field)(*args))
        for precision, tol in (('double', 1e-10), ('single', 3e-6 if shape not in ('sparse', 'wide patch') else 5e-5)):
            got = np.stack(getattr(made[1], field)(*args, precision=precision))
            assert np.abs(got - want).max() <= tol * np.abs(want).max(), (field, precision)


def test_fp64_phases_of_columns_far_out(gpu):
    """A discrete plane wave at azimuth 0 on columns 30 to 60 um out and up to 30 um high: kappa x and k_z z are
    products of FP64 numbers, and their phases, several hundred radians, keep an absolute error of a few 1e-16 (not of
    their own size, 1e-13)."""
    from smuthi_amd.expansions import PlaneWaveExpansion
    x, z = np.meshgrid([30123.4, -44567.8, 59876.5], np.linspace(100.0, 30000.0, 40))
    x, z = x.ravel(), z.ravel()
    for kappa in K * np.array([0.31, 0.64, 0.977]):
        pwe = PlaneWaveExpansion(K, [kappa], [0.0], 'upgoing', [0, 0, 0], 0, np.inf)
        pwe.coefficients[0] = 0.8 - 0.3j
        got = pwe.electric_field(x, np.zeros_like(x), z, precision='double')[1]
        phase = np.longdouble(kappa) * x.astype(np.longdouble) + \
            np.longdouble(pwe.k_z()[0].real) * z.astype(np.longdouble)
        want = (0.8 - 0.3j) * (np.cos(phase) + 1j * np.sin(phase)).astype(complex)
        assert np.linalg.norm(got - want) <= 2e-15 * np.linalg.norm(want)
