"""The factorisation behind the explicit matrix's direct solve, at the sizes
where it can go wrong: less than one panel of columns, a last panel that is not
full, 1024 rows and just over (one or two rows per thread), the largest matrix
it takes and the next one (the library's), against the definition of M = 1 -
diag(t) W in numpy. T is large and uneven, so most pivots lie off the diagonal.
Partial pivoting is backward stable: the residual of n unknowns stays below a
few n 1e-16 of |M| |x| + |b| for every right-hand side."""
import numpy as np
import pytest

from test_gpu_explicit_batch import _operator

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def gpu():
    from smuthi_amd import cuda
    assert cuda.enable_gpu(), 'MI355X not available'
    return cuda


# unknowns: 6, 12, 210, 1020, 1026, 2046, 2052
@pytest.mark.parametrize('n,l_max', [(1, 1), (2, 1), (7, 3), (34, 3), (171, 1), (341, 1), (342, 1)])
def test_direct_solve_is_backward_stable(gpu, n, l_max):
    op = _operator(n, l_max)
    W = op.coupling_matrix
    size = len(W)
    print('LU: %d unknowns' % size, flush=True)
    rng = np.random.default_rng(n)
    t = 10 ** rng.uniform(-1, 2, size) / np.abs(W).max() * np.exp(2j * np.pi * rng.uniform(size=size))
    M = np.eye(size) - t[:, None] * W
    b = rng.standard_normal((2, size)) + 1j * rng.standard_normal((2, size))
    x = op.solve_master(t, b, 1e-6, precision='lu')
    for v, r in zip(x, b):
        res = np.abs(M @ v - r).max()
        assert res <= 4e-16 * size * (np.abs(M).sum(1).max() * np.abs(v).max() + np.abs(r).max()), res


def test_weak_coupling_leaves_the_identity_unrounded(gpu):
    """M = 1 - diag(t) W with a coupling of 1e-3, 1800 unknowns: the updates of the trailing matrix round its coupling,
    not the 1s of its diagonal. What is left are the substitutions' roundings of x, 6.0e-16 (the library's whole solve:
    6.3e-16); rounding the 1s once per eight columns adds sqrt(225 / 12) 1.1e-16, 8.1e-16 in all."""
    op = _operator(60, 3)
    W = op.coupling_matrix
    size = len(W)
    errors = []
    for seed in range(3):
        rng = np.random.default_rng(seed)
        t = 1e-3 / np.linalg.norm(W, 'fro') * np.exp(2j * np.pi * rng.uniform(size=size))
        b = rng.standard_normal(size) + 1j * rng.standard_normal(size)
        x = op.solve_master(t, b, 1e-6, precision='lu')
        # Neumann series with 64-bit mantissas: |t W| <= 1e-3, so six terms leave 1e-18
        tl, Wl = t.astype(np.clongdouble), W.astype(np.clongdouble)
        want = term = b.astype(np.clongdouble)
        for _ in range(6):
            term = tl * (Wl @ term)
            want = want + term
        errors.append(float(np.linalg.norm((x - want).astype(complex)) / np.linalg.norm(b)))
    print('LU of weak coupling: errors', errors, flush=True)
    assert max(errors) <= 7e-16
