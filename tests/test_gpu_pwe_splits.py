"""Scattered-field assembly with its particles split over workgroups: one particle,
whole chunks of 32, one more and one less, many chunks at one direction
(extinction) and at many, several chunks in one workgroup, orders in one and in several launches, against a plain numpy sum of the
same formula at 64 bits. FP64 sums of n terms differ by about n 1e-16 of the
largest; FP32 rounds coefficients, phases and sums to 6e-8 each, 5e-5 as the
assembly's own tests."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

K = 2 * np.pi / 550


@pytest.mark.parametrize('n,n_k,n_a,l_max', [(1, 1, 1, 1), (64, 3, 70, 2), (65, 1, 1, 3), (700, 1, 1, 3),
                                             (700, 2, 300, 1), (130, 2, 9, 6), (31, 1, 5, 2),
                                             (32, 2, 40, 3), (33, 3, 17, 1)])
def test_assembly_matches_numpy(n, n_k, n_a, l_max):
    from smuthi_amd import _lib, cuda, fields
    assert cuda.enable_gpu(), 'MI355X not available'
    rng = np.random.default_rng(n + n_k + l_max)
    B = fields.blocksize(l_max, l_max)
    _, _, m = fields.index_arrays(l_max, l_max)
    xyz = np.stack([rng.uniform(-2000, 2000, n), rng.uniform(-2000, 2000, n), rng.uniform(50, 300, n)], 1)
    kp = (K * rng.uniform(0, 1.4, n_k) - 1j * K * 0.01 * rng.integers(0, 2, n_k)).astype(complex)
    kz = fields.k_z(k_parallel=kp, k=K).astype(complex)
    al = np.sort(rng.uniform(0, 2 * np.pi, n_a))

    def c(*s):
        return np.ascontiguousarray(rng.standard_normal(s) + 1j * rng.standard_normal(s))
    coef, btab = c(n, B), c(n_k, 2, 2, B)
    z_ref = 20.0
    want = np.zeros((2, 2, n_k, n_a), complex)
    for k in range(n_k):
        ph = np.exp(-1j * kp[k] * (xyz[:, :1] * np.cos(al) + xyz[:, 1:2] * np.sin(al)))
        for d, s in ((0, 1), (1, -1)):
            b = coef * np.exp(1j * s * kz[k] * (z_ref - xyz[:, 2]))[:, None]
            for pol in range(2):
                want[d, pol, k] = ((b * btab[k, d, pol]).T @ ph * np.exp(1j * m[:, None] * al)).sum(0)
    print('assembly: %d particles, %d x %d waves' % (n, n_k, n_a), flush=True)
    for prec, tol in ((_lib.FP64, 1e-11), (_lib.FP32, 5e-5)):
        got = np.zeros_like(want)
        ms = ctypes.c_double()
        _lib.check(_lib.load().smh_pwe_assemble(cuda.context(), n, _lib.dptr(xyz), l_max, l_max, _lib.dptr(coef), z_ref,
                                                n_k, _lib.dptr(kp), _lib.dptr(kz), _lib.dptr(btab), n_a, _lib.dptr(al),
                                                _lib.dptr(got), prec, ctypes.byref(ms)), cuda.context(), 'assemble')
        assert np.abs(got - want).max() <= tol * np.abs(want).max()


@pytest.mark.parametrize('n,l_max', [(101, 3), (300, 1)])
def test_workgroups_of_several_chunks(n, l_max):
    """As many waves as fill the chip, so that one workgroup goes through all particles: three chunks of 32 and five
    more, and nine and twelve more with FP32 sums put away in between; a few of the kappa are checked."""
    from smuthi_amd import _lib, cuda, fields
    assert cuda.enable_gpu(), 'MI355X not available'
    rng = np.random.default_rng(n)
    n_k, n_a = 700, 400
    B = fields.blocksize(l_max, l_max)
    _, _, m = fields.index_arrays(l_max, l_max)
    xyz = np.stack([rng.uniform(-2000, 2000, n), rng.uniform(-2000, 2000, n), rng.uniform(50, 300, n)], 1)
    kp = (K * rng.uniform(0, 1.4, n_k) - 1j * K * 0.01 * (np.arange(n_k) % 2)).astype(complex)
    kz = fields.k_z(k_parallel=kp, k=K).astype(complex)
    al = np.sort(rng.uniform(0, 2 * np.pi, n_a))

    def c(*s):
        return np.ascontiguousarray(rng.standard_normal(s) + 1j * rng.standard_normal(s))
    coef, btab = c(n, B), c(n_k, 2, 2, B)
    z_ref = 20.0
    print('assembly: %d particles, %d x %d waves' % (n, n_k, n_a), flush=True)
    for prec, tol in ((_lib.FP64, 1e-11), (_lib.FP32, 5e-5)):
        got, ms = np.zeros((2, 2, n_k, n_a), complex), ctypes.c_double()
        _lib.check(_lib.load().smh_pwe_assemble(cuda.context(), n, _lib.dptr(xyz), l_max, l_max, _lib.dptr(coef), z_ref,
                                                n_k, _lib.dptr(kp), _lib.dptr(kz), _lib.dptr(btab), n_a, _lib.dptr(al),
                                                _lib.dptr(got), prec, ctypes.byref(ms)), cuda.context(), 'assemble')
        for k in (0, 1, 350, 698, 699):
            ph = np.exp(-1j * kp[k] * (xyz[:, :1] * np.cos(al) + xyz[:, 1:2] * np.sin(al)))
            for d, s in ((0, 1), (1, -1)):
                b = coef * np.exp(1j * s * kz[k] * (z_ref - xyz[:, 2]))[:, None]
                want = np.stack([((b * btab[k, d, pol]).T @ ph * np.exp(1j * m[:, None] * al)).sum(0)
                                 for pol in range(2)])
                assert np.abs(got[d, :, k] - want).max() <= tol * np.abs(want).max(), (prec, k, d)


def test_fp64_phases_over_a_wide_array():
    """One particle 41 um out at azimuth 0, where kappa x is a product of two FP64 numbers: its phase, some 600
    radians, keeps an absolute error of a few 1e-16 (not of its own size, 7e-14)."""
    from smuthi_amd import _lib, cuda, fields
    assert cuda.enable_gpu(), 'MI355X not available'
    rng = np.random.default_rng(2)
    n_k = 200
    B = fields.blocksize(1, 1)
    _, _, m = fields.index_arrays(1, 1)
    xyz, z_ref = np.array([[41234.567, 0.0, 100.0]]), 100.0
    kp = (K * rng.uniform(0.5, 1.4, n_k)).astype(complex)
    kz = fields.k_z(k_parallel=kp, k=K).astype(complex)

    def c(*s):
        return np.ascontiguousarray(rng.standard_normal(s) + 1j * rng.standard_normal(s))
    coef, btab, al = c(1, B), c(n_k, 2, 2, B), np.zeros(1)
    got, ms = np.zeros((2, 2, n_k, 1), complex), ctypes.c_double()
    _lib.check(_lib.load().smh_pwe_assemble(cuda.context(), 1, _lib.dptr(xyz), 1, 1, _lib.dptr(coef), z_ref, n_k,
                                            _lib.dptr(kp), _lib.dptr(kz), _lib.dptr(btab), 1, _lib.dptr(al),
                                            _lib.dptr(got), _lib.FP64, ctypes.byref(ms)), cuda.context(), 'assemble')
    phase = kp.real.astype(np.longdouble) * np.longdouble(xyz[0, 0])
    wave = (np.cos(phase) - 1j * np.sin(phase)).astype(complex)
    want = (btab @ coef[0]).transpose(1, 2, 0) * wave
    assert np.linalg.norm(got[..., 0] - want) <= 2e-15 * np.linalg.norm(want)


def test_fp32_keeps_its_digits_over_many_particles():
    """4000 particles over 60 um that one workgroup sums (the waves alone fill the chip), lossless and lossy
    kappa. Coefficients, phases (native sine and cosine, 1e-7) and the sums of 128 particles are rounded to 32
    bits, independently per particle: 2e-7 to 3e-7 of the result whatever their number; 6e-7 with room."""
    from smuthi_amd import _lib, cuda, fields
    assert cuda.enable_gpu(), 'MI355X not available'
    rng = np.random.default_rng(7)
    n, n_k, n_a, l_max = 4000, 700, 400, 2
    B = fields.blocksize(l_max, l_max)
    _, _, m = fields.index_arrays(l_max, l_max)
    xyz = np.stack([rng.uniform(-3e4, 3e4, n), rng.uniform(-3e4, 3e4, n), rng.uniform(50, 300, n)], 1)
    kp = (K * rng.uniform(0.1, 1.4, n_k) - 1j * K * 0.01 * (np.arange(n_k) % 2)).astype(complex)
    kz = fields.k_z(k_parallel=kp, k=K).astype(complex)
    al = np.linspace(0, 2 * np.pi, n_a)

    def c(*s):
        return np.ascontiguousarray(rng.standard_normal(s) + 1j * rng.standard_normal(s))
    coef, btab = c(n, B), c(n_k, 2, 2, B)
    z_ref = 20.0
    got, ms = np.zeros((2, 2, n_k, n_a), complex), ctypes.c_double()
    print('assembly: %d particles, %d x %d waves' % (n, n_k, n_a), flush=True)
    _lib.check(_lib.load().smh_pwe_assemble(cuda.context(), n, _lib.dptr(xyz), l_max, l_max, _lib.dptr(coef), z_ref,
                                            n_k, _lib.dptr(kp), _lib.dptr(kz), _lib.dptr(btab), n_a, _lib.dptr(al),
                                            _lib.dptr(got), _lib.FP32, ctypes.byref(ms)), cuda.context(), 'assemble')
    for k in (0, 1, 350, 699):
        ph = np.exp(-1j * kp[k] * (xyz[:, :1] * np.cos(al) + xyz[:, 1:2] * np.sin(al)))
        for d, s in ((0, 1), (1, -1)):
            b = coef * np.exp(1j * s * kz[k] * (z_ref - xyz[:, 2]))[:, None]
            for pol in range(2):
                want = ((b * btab[k, d, pol]).T @ ph * np.exp(1j * m[:, None] * al)).sum(0)
                err = np.linalg.norm(got[d, pol, k] - want) / np.linalg.norm(want)
                assert err <= 6e-7, (k, d, pol, err)
