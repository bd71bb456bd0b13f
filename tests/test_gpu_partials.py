"""Work items and the reduction of their partial sums at the sizes where their
rules change: receiver chunks that end at a chunk's limit, just after it and
evened over two chunks, one or several strands per result, the one-launch
input bound and the two-pass one. A smooth synthetic table keeps the reference
(plain numpy, linear interpolation, FP64) cheap at thousands of particles.

Tolerances: FP64 sums of n terms of similar size in another order differ by
about sqrt(n) 1e-16 of the largest row, 1e-13 leaves room at n = 2740; the
FP32 results round tap values, phases and products to 2^-24, a few of them per
term and averaging over the terms, 2e-6 as in the oracle tests."""
import numpy as np
import pytest

from smuthi_amd.particles import Sphere

pytestmark = pytest.mark.gpu

H = 40.0


@pytest.fixture(scope='module')
def gpu():
    from smuthi_amd import cuda
    assert cuda.enable_gpu(), 'MI355X not available'
    return cuda


def _system(n, seed):
    rng = np.random.default_rng(seed)
    m = int(np.ceil(np.sqrt(n)))
    site = rng.permutation(m * m)[:n]
    xy = np.stack([site % m, site // m], 1) * 300.0 + rng.uniform(-50, 50, (n, 2))
    rho_max = np.hypot(*(xy.max(0) - xy.min(0)))
    rho = np.arange(-3 * H, rho_max + 3 * H, H)
    a, p = rng.uniform(0.5, 1.5, (6, 6)), rng.uniform(0, 2 * np.pi, (6, 6))
    table = a * np.exp(1j * (0.004 * rho[:, None, None] + p)) / (1 + np.abs(rho[:, None, None]) / 500)
    return xy, rho, table


def _reference(xy, rho, table, x):
    """x [nrhs, n, 6]; linear interpolation between the table rows, phases e^{i (m2 - m1) phi}."""
    m = np.tile([-1, 0, 1], 2)
    y = np.zeros_like(x)
    for i in range(len(xy)):
        d = xy[i] - xy
        t = (np.hypot(d[:, 0], d[:, 1]) - rho[0]) / H
        r = np.floor(t).astype(int)
        w = (t - r)[:, None, None]
        e = np.exp(1j * np.arctan2(d[:, 1], d[:, 0])[:, None] * m)
        L = (1 - w) * table[r] + w * table[r + 1]
        y[:, i] = np.einsum('jk,rjk->rk', e.conj(), np.einsum('jkl,rjl->rjk', L, e[None] * x))
    return y


@pytest.mark.parametrize('n', [2, 17, 511, 513, 2740])
def test_partial_sums_match_reference(gpu, n):
    from smuthi_amd.linear_system import CouplingMatrixRadialLookupCUDA
    xy, rho, table = _system(n, n)
    parts = [Sphere([a, b, 200.0], 1.5, 50.0, 1, 1) for a, b in xy]
    op = CouplingMatrixRadialLookupCUDA.from_table(table, rho, parts, H, 'linear')
    rng = np.random.default_rng(n)
    x = rng.standard_normal((9, n * 6)) + 1j * rng.standard_normal((9, n * 6))
    want = _reference(xy, rho, table, x.reshape(9, n, 6)).reshape(9, -1)
    print('partials: %d particles' % n, flush=True)
    for precision, tol in (('double', 1e-13), ('single', 2e-6), ('half', 2e-3)):
        got = op.matvec(x, precision)  # a full and a nearly empty batch
        assert np.linalg.norm(got - want) <= tol * np.linalg.norm(want), (precision, 'batch')
        if precision != 'half':
            got = op.matvec(x[0], precision)
            assert np.linalg.norm(got - want[0]) <= tol * np.linalg.norm(want[0]), (precision, 'single')
