"""The volume lookup's matvecs for several right-hand sides (cubic: pairs sorted
by bin, products summed per receiver in slabs; bilinear: receiver chunks)
against its single-vector FP64 matvec, over every block shape (one to three
tiles per row group, rows with and without spline moments) and where the walk can go
wrong: one particle, odd numbers of pairs in a bin, many pairs in a bin (two
heights), several slabs (420 particles: 176 k pairs, a slab holds 131 k of them
in FP32 and 65 k in FP64), ensembles of different sizes.

Tolerances: both FP64 kernels add the same products of the same taps in another
order, sqrt(n taps) 1e-16 of the result, 1e-12 with room. FP32 rounds weights,
taps, phases and products to 2^-24, some of each per term, averaged over the
terms: 3e-6 as in the oracle tests. FP16 operands: 2^-11 per operand, 3e-3 as
there."""
import ctypes

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


def _ensembles(offsets):
    """Class of volume operators over the ensembles of particles [offsets[e], offsets[e + 1])."""
    from smuthi_amd import _lib, cuda
    from smuthi_amd.volume import CouplingMatrixVolumeLookupCUDA

    class Ensembles(CouplingMatrixVolumeLookupCUDA):
        def _create(self, xyz):
            off = np.ascontiguousarray(offsets, dtype=np.int64)
            self._op = ctypes.c_void_p()
            _lib.check(_lib.load().smh_volume_create_ensembles(
                cuda.context(), len(off) - 1, off.ctypes.data_as(ctypes.POINTER(ctypes.c_int64)), _lib.dptr(xyz),
                _lib.iptr(self._lmax), _lib.iptr(self._mmax), self.l_max, self.m_max, float(self.rho_array[0]),
                float(self.sum_z_array[0]), float(self.diff_z_array[0]), float(self.resolution), len(self.rho_array),
                len(self.sum_z_array), self._interp, ctypes.byref(self._op)), cuda.context(), 'create')
    return Ensembles


def _operator(n, l_max, m_max, kind, heights, seed, size=1.0, zero_below=0.0, offsets=None):
    from smuthi_amd.volume import CouplingMatrixVolumeLookupCUDA
    make = CouplingMatrixVolumeLookupCUDA if offsets is None else _ensembles(offsets)
    rng = np.random.default_rng(seed)
    m = int(np.ceil(np.sqrt(n)))
    site = rng.permutation(m * m)[:n]
    xy = np.stack([site % m, site // m], 1) * 60.0 + rng.uniform(-10, 10, (n, 2))
    z = rng.uniform(150, 300, n) if heights is None else rng.choice(heights, n)
    parts = [Sphere([a, b, c], 1.5, 50.0, l_max, m_max) for (a, b), c in zip(xy, z)]
    rho = np.arange(-3 * H, np.hypot(*np.ptp(xy, axis=0)) + 5 * H, H)
    sz = np.arange(300 - 4 * H, 600 + 5 * H, H)
    dz = np.arange(-150 - 4 * H, 150 + 5 * H, H)
    B = 2 * (m_max * (m_max + 2) + (l_max - m_max) * (2 * m_max + 1))

    # smooth along rho and z, entries of different size
    def table(zs):
        a, p, k = rng.uniform(0.1, 1.5, (B, B)), rng.uniform(0, 2 * np.pi, (B, B)), rng.uniform(-1, 1, (B, B))
        r = rho[:, None, None, None]
        t = size * a * np.exp(1j * (0.004 * r + 0.003 * k * zs[None, :, None, None] + p)) / (1 + np.abs(r) / 500)
        return t * (np.abs(r) >= zero_below)
    kw = {'linear': dict(interpolator_kind='linear'),
          'catmull-rom': dict(interpolator_kind='cubic', cubic_interpolant='catmull-rom'),
          'spline': dict(interpolator_kind='cubic', cubic_interpolant='spline')}[kind]
    return make.from_tables(table(sz), table(dz), rho, sz, dz, parts, H, **kw), rng


@pytest.mark.parametrize('n,l_max,m_max,kind,heights', [
    (1, 1, 1, 'linear', None), (2, 2, 2, 'spline', None), (37, 2, 1, 'catmull-rom', None),
    (64, 3, 3, 'linear', (160.0, 200.0)), (17, 3, 3, 'spline', None), (23, 3, 2, 'catmull-rom', None),
    (33, 3, 1, 'spline', (160.0, 200.0)), (12, 4, 4, 'catmull-rom', None), (11, 4, 3, 'spline', None),
    (9, 4, 2, 'linear', None), (420, 1, 1, 'spline', None)])
def test_batched_matvecs_match_single_vector(gpu, n, l_max, m_max, kind, heights):
    op, rng = _operator(n, l_max, m_max, kind, heights, n + l_max)
    size = op.shape[0]
    for nrhs in (8, 3):
        V = rng.standard_normal((nrhs, size)) + 1j * rng.standard_normal((nrhs, size))
        V[-1] *= 1e-3
        want = np.stack([op.matvec(v, 'double') for v in V])
        scale = np.linalg.norm(want, axis=1)
        for precision, tol in (('double', 1e-12), ('single', 3e-6), ('half', 3e-3)):
            got = op.matvec(V, precision)
            err = np.linalg.norm(got - want, axis=1) / scale
            # (FP16 operands share one scale over the right-hand sides)
            err = err[:-1] if precision == 'half' else err
            assert err.max() < tol, (precision, err)
            # cubic: sums in a fixed order, the same to the last bit
            assert kind == 'linear' or np.array_equal(got, op.matvec(V, precision))


@pytest.mark.parametrize('kind,l_max', [('linear', 2), ('catmull-rom', 3), ('spline', 1)])
def test_ensembles_of_different_sizes(gpu, kind, l_max):
    """Pairs of one ensemble only: one operator over 1, 37, 2 and 60 particles against the operator over all hundred,
    applied to the vectors of one ensemble at a time."""
    off = [0, 1, 38, 40, 100]
    op, rng = _operator(100, l_max, l_max, kind, None, 9, offsets=off)
    whole, _ = _operator(100, l_max, l_max, kind, None, 9)
    B = op.blocksize
    V = rng.standard_normal((8, op.shape[0])) + 1j * rng.standard_normal((8, op.shape[0]))
    want = np.zeros_like(V)
    for a, b in zip(off[:-1], off[1:]):
        part = np.zeros_like(V)
        part[:, a * B:b * B] = V[:, a * B:b * B]
        want[:, a * B:b * B] = np.stack([whole.matvec(v, 'double') for v in part])[:, a * B:b * B]
    for precision, tol in (('double', 1e-12), ('single', 3e-6), ('half', 3e-3)):
        got = op.matvec(V, precision)
        for a, b in zip(off[:-1], off[1:]):
            g, w = got[:, a * B:b * B], want[:, a * B:b * B]
            assert np.linalg.norm(g - w) < tol * np.linalg.norm(w), (precision, a)


@pytest.mark.parametrize('kind', ['linear', 'catmull-rom', 'spline'])
@pytest.mark.parametrize('size', [1.0, 1e-2, 1e-4])
def test_half_next_to_rows_of_zeros(gpu, kind, size):
    """Table nodes at small distances hold zeros (no pair is that close), and the pairs next to them interpolate
    with them: the FP16 error is that of the other pairs, whatever the size of the table's values. 2^-11 per
    operand, averaged over the terms: 4e-4 without rows of zeros, 1e-3 with room."""
    op, rng = _operator(60, 3, 3, kind, None, 3, size, zero_below=70.0)
    V = rng.standard_normal((8, op.shape[0])) + 1j * rng.standard_normal((8, op.shape[0]))
    want = op.matvec(V, 'double')
    assert np.linalg.norm(op.matvec(V, 'half') - want) < 1e-3 * np.linalg.norm(want)


@pytest.mark.parametrize('kind,grouped', [('linear', True), ('spline', False), ('catmull-rom', False)])
def test_autotune_times_one_launch_once(gpu, kind, grouped):
    """The slab kernels have no launch shapes to choose from: every candidate has the one launch's time, and the
    first is named. The single-vector and bilinear kernels are timed candidate by candidate."""
    op, rng = _operator(60, 2, 2, kind, None, 5)
    V = rng.standard_normal((8, op.shape[0])) + 1j * rng.standard_normal((8, op.shape[0]))
    cand = [(4, 0), (16, 1), (8, 0), (32, 1), (16, 0)]
    for precision in ('half', 'single', 'double'):
        before = op.matvec(V, precision)
        res = op.autotune(batch=True, precision=precision, iters=2, candidates=cand)
        times = set(res['matvec_ms'].values())
        assert min(times) > 0
        if grouped:
            assert len(times) > 1
        else:
            assert len(times) == 1 and res['best'] == cand[0]
            assert np.array_equal(op.matvec(V, precision), before)
    assert len(set(op.autotune(batch=False, precision='single', iters=2, candidates=cand)['matvec_ms'].values())) > 1
