"""Products of the explicit matrix with blocks of vectors (the MFMA kernel) and
the block solves on it, at sizes below one turn of columns, at whole turns and
with columns and rows left over, for full and nearly empty blocks, against
numpy on the downloaded matrix. FP64 products of n terms in another order
differ by about n 1e-16; the FP32 ones carry the complex64 rounding of the
matrix and the vectors (6e-8 each, averaging) and FP32 sums, 2e-6 as the
single-vector product's test."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

WL = 550.0


@pytest.fixture(scope='module')
def gpu():
    from smuthi_amd import cuda
    assert cuda.enable_gpu(), 'MI355X not available'
    return cuda


def _operator(n, l_max):
    from smuthi_amd import fields
    from smuthi_amd.layers import LayerSystem
    from smuthi_amd.linear_system import CouplingMatrixExplicit
    from smuthi_amd.particles import Sphere
    rng = np.random.default_rng(n)
    m = int(np.ceil(np.sqrt(n)))
    parts = [Sphere([260.0 * (i % m), 260.0 * (i // m), 150 + 60 * rng.uniform()], 1.6 + 0.02j, 80, l_max, l_max)
             for i in range(n)]
    kp = fields.reasonable_Sommerfeld_kpar_contour(WL, layer_refractive_indices=[1.5, 1], neff_resolution=3e-2)
    return CouplingMatrixExplicit(WL, parts, LayerSystem([0, 0], [1.5, 1]), k_parallel=kp)


# unknowns: 6, 32 columns short of two turns, 96 = whole turns, 102, 210, 1050
@pytest.mark.parametrize('n,l_max', [(1, 1), (10, 1), (16, 1), (17, 1), (7, 3), (35, 3)])
def test_block_products_and_solves(gpu, n, l_max):
    op = _operator(n, l_max)
    W = op.coupling_matrix
    rng = np.random.default_rng(n + 1)
    x = rng.standard_normal((9, len(W))) + 1j * rng.standard_normal((9, len(W)))
    want = x @ W.T
    print('explicit blocks: %d unknowns' % len(W), flush=True)
    for precision, tol in (('double', 1e-13), ('single', 2e-6)):
        got = op.matvec(x, precision)
        for g, w in zip(got, want):
            assert np.linalg.norm(g - w) <= tol * np.linalg.norm(w), precision
    t = 0.2 / max(1.0, np.abs(W).sum(1).max()) * np.exp(2j * np.pi * rng.uniform(size=len(W)))
    exact = np.linalg.solve(np.eye(len(W)) - t[:, None] * W, x.T).T
    for precision in ('double', 'mixed'):
        got, stats, ok = op.solve_master(t, x, 1e-10, precision=precision, with_stats=True)
        assert ok and stats['relative_residual'] <= 1e-10
        assert np.linalg.norm(got - exact) <= 1e-9 * np.linalg.norm(exact), precision


@pytest.mark.parametrize('n,l_max', [(20, 2), (20, 3), (60, 3)])
def test_block_products_are_as_accurate_as_single_ones(gpu, n, l_max):
    """Errors against 64-bit mantissas of a block product and of the same vectors one by one (sums of a wavefront: a
    few terms per lane and a tree). FP32 blocks gather their chains in FP64, 0.5 to 0.7 of the single vectors' error;
    FP64 blocks have chains and trees of the same length, 0.7 to 1.01 of it, 1.08 with room."""
    op = _operator(n, l_max)
    W = op.coupling_matrix
    rng = np.random.default_rng(3)
    x = rng.standard_normal((8, len(W))) + 1j * rng.standard_normal((8, len(W)))
    want = np.stack([W.astype(np.clongdouble) @ v.astype(np.clongdouble) for v in x])

    def error(y):
        return float(np.linalg.norm((y - want).astype(complex)) / np.linalg.norm(want.astype(complex)))
    for precision, bound in (('single', 0.9), ('double', 1.08)):
        block, single = error(op.matvec(x, precision)), error(np.stack([op.matvec(v, precision) for v in x]))
        print('explicit blocks: %d unknowns, %s: %.2e, one by one %.2e' % (len(W), precision, block, single), flush=True)
        assert block <= bound * single, precision


def test_explicit_operator_refuses_what_it_did(gpu):
    from smuthi_amd._lib import SmhError
    from smuthi_amd.batch import set_preconditioner
    op = _operator(3, 1)
    x = np.ones((3, op.shape[0]), complex)
    with pytest.raises(SmhError):
        op.matvec(x, 'half')
    with pytest.raises(SmhError):
        op.bench_matvec_batch('single', iters=1)
    with pytest.raises(SmhError):
        op.autotune()
    with pytest.raises(SmhError):
        set_preconditioner(op, np.zeros((3, 6, 6), complex))
    with pytest.raises(SmhError):
        op.solve_master(np.full(op.shape[0], 0.1), x, 1e-6, precision='mixed16')


def test_each_right_hand_side_of_a_block_has_its_own_steps(gpu):
    """maxiter counts the steps of each right-hand side, as if it were solved alone. Noise takes most steps, in one
    sweep of the refinement; an eigenvector with 1e-6 of noise few, in two. Together the second sweeps follow the
    longest first one, and the block still passes with the steps that its longest member takes alone."""
    op = _operator(24, 2)
    W = op.coupling_matrix
    n, tol = len(W), 1.5e-7
    rng = np.random.default_rng(5)
    t = 0.8 / np.abs(np.linalg.eigvals(W)).max() * np.exp(2j * np.pi * rng.uniform(size=n))
    _, vec = np.linalg.eig(np.eye(n) - t[:, None] * W)

    def noise():
        v = rng.standard_normal(n) + 1j * rng.standard_normal(n)
        return v / np.linalg.norm(v)

    def alone(x):
        return [op.solve_master(t, v, tol, precision='mixed', restart=100, with_stats=True)[1] for v in x]
    hard, easy = [noise() for _ in range(24)], [vec[:, 3 * j] + 1e-6 * noise() for j in range(24)]
    sh, se = alone(hard), alone(easy)
    one = [(s['iterations'], j) for j, s in enumerate(sh) if s['sweeps'] == 1 and s['relative_residual'] < 0.85 * tol]
    steps, j = max(one)
    two = [k for k, s in enumerate(se) if s['sweeps'] == 2 and s['iterations'] < steps][:7]
    print('steps alone %d, %s' % (steps, [se[k]['iterations'] for k in two]), flush=True)
    assert len(two) == 7
    x = np.stack([hard[j]] + [easy[k] for k in two])
    got, stats, ok = op.solve_master(t, x, tol, precision='mixed', restart=100, maxiter=steps, with_stats=True)
    assert ok and stats['relative_residual'] <= tol and stats['iterations'] > steps, stats
    assert not op.solve_master(t, x, tol, precision='mixed', restart=100, maxiter=steps // 2, with_stats=True)[2]
