"""Solves of one right-hand side on the device: systems whose Arnoldi step runs
in one workgroup (up to 4096 unknowns, edge at 682 / 683 particles of 6, and up
to 64 steps of 4092), the several-launch step above, restart lengths from one step to the largest basis,
and repeated solves (the first runs eagerly, the second captures its graphs,
the third replays them, with eager matvecs between), and solves of different
operators by several threads on the context's one stream, while graphs are
captured. The residual is taken
with the plain numpy operator of the partial-sum tests; an FP64 solve to tol
leaves tol plus the FP64 operators' own difference (1e-13)."""
import ctypes
import threading

import numpy as np
import pytest

from smuthi_amd.particles import Sphere
from test_gpu_partials import H, _reference, _system

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def gpu():
    from smuthi_amd import cuda
    assert cuda.enable_gpu(), 'MI355X not available'
    return cuda


@pytest.mark.parametrize('n,restart', [(2, 1), (17, 127), (682, 6), (682, 40), (683, 6), (683, 40)])
def test_single_solves_meet_the_tolerance(gpu, n, restart):
    from smuthi_amd.linear_system import CouplingMatrixRadialLookupCUDA
    xy, rho, table = _system(n, n)
    op = CouplingMatrixRadialLookupCUDA.from_table(table, rho, [Sphere([a, b, 200.0], 1.5, 50.0, 1, 1)
                                                                for a, b in xy], H, 'linear')
    rng = np.random.default_rng(n + restart)
    d = np.hypot(xy[:, None, 0] - xy[None, :, 0], xy[:, None, 1] - xy[None, :, 1])
    t = (0.25 / (6 * (1 / (1 + d / 500)).sum(1).max()) * np.exp(2j * np.pi * rng.uniform(size=(n, 6)))).ravel()
    b = rng.standard_normal(n * 6) + 1j * rng.standard_normal(n * 6)
    print('single solve: %d particles, restart %d' % (n, restart), flush=True)
    first = None
    for repeat in range(3):
        for precision in ('double', 'mixed'):
            x, stats, ok = op.solve_master(t, b, 1e-9, precision=precision, restart=restart, with_stats=True)
            assert ok and stats['relative_residual'] <= 1e-9
            r = b - x + t * _reference(xy, rho, table, x.reshape(1, n, 6)).ravel()
            assert np.linalg.norm(r) <= (1e-9 + 1e-12) * np.linalg.norm(b), (precision, repeat)
            first = x if first is None else first
            assert np.linalg.norm(x - first) <= 1e-8 * np.linalg.norm(first)
        op.matvec(b, 'single')


def test_steps_on_both_sides_of_the_basis_limit(gpu):
    """A cycle of 100 steps that does not converge: the first 64 run in one workgroup, the others in several
    launches. Its residual is the true one of its solution, and the smallest over the same Krylov space that a block
    solve (several launches throughout) finds, up to the FP64 roundings of 100 steps on a basis orthogonalised twice
    (100 x 1e-16 x the growth of |x| over |b|, below 1e-9)."""
    from smuthi_amd.linear_system import CouplingMatrixRadialLookupCUDA
    n = 682
    xy, rho, table = _system(n, n)
    op = CouplingMatrixRadialLookupCUDA.from_table(table, rho, [Sphere([a, b, 200.0], 1.5, 50.0, 1, 1)
                                                                for a, b in xy], H, 'linear')
    rng = np.random.default_rng(1)
    d = np.hypot(xy[:, None, 0] - xy[None, :, 0], xy[:, None, 1] - xy[None, :, 1])
    t = (4000 / (6 * (1 / (1 + d / 500)).sum(1).max()) * np.exp(2j * np.pi * rng.uniform(size=(n, 6)))).ravel()
    b = rng.standard_normal((2, n * 6)) + 1j * rng.standard_normal((2, n * 6))
    kw = dict(precision='double', restart=100, maxiter=100, with_stats=True)
    worst = []
    for repeat in range(3):
        alone = [op.solve_master(t, v, 1e-12, **kw) for v in b]
        for (x, stats, ok), v in zip(alone, b):
            res = np.linalg.norm(v - x + t * _reference(xy, rho, table, x.reshape(1, n, 6)).ravel())
            assert not ok and stats['iterations'] == 100
            assert abs(res / np.linalg.norm(v) - stats['relative_residual']) <= 1e-9
        worst.append(max(s['relative_residual'] for _, s, _ in alone))
    block = op.solve_master(t, b, 1e-12, **kw)[1]['relative_residual']
    assert np.abs(np.array(worst) / block - 1).max() <= 1e-6, (worst, block)


def test_shorter_restarts_keep_the_workspace(gpu):
    """Restart lengths in turn, eager, captured and replayed: the arrays of the longest serve the shorter ones, so
    no device memory is given back (5000 unknowns: 10 MB of basis at 120, 0.6 MB at 6)."""
    from smuthi_amd.linear_system import CouplingMatrixRadialLookupCUDA
    hip = ctypes.CDLL('libamdhip64.so')

    def free_memory():
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value
    n = 834
    xy, rho, table = _system(n, n)
    op = CouplingMatrixRadialLookupCUDA.from_table(table, rho, [Sphere([a, b, 200.0], 1.5, 50.0, 1, 1)
                                                                for a, b in xy], H, 'linear')
    rng = np.random.default_rng(3)
    d = np.hypot(xy[:, None, 0] - xy[None, :, 0], xy[:, None, 1] - xy[None, :, 1])
    t = (0.25 / (6 * (1 / (1 + d / 500)).sum(1).max()) * np.exp(2j * np.pi * rng.uniform(size=(n, 6)))).ravel()
    b = rng.standard_normal((3, n * 6)) + 1j * rng.standard_normal((3, n * 6))
    for rhs in (b[0], b):
        op.solve_master(t, rhs, 1e-9, precision='double', restart=120)
        free = free_memory()
        for restart in (6, 120, 2, 6, 120, 6):
            x = op.solve_master(t, rhs, 1e-9, precision='double', restart=restart)
            for v, r in zip(x.reshape(-1, n * 6), rhs.reshape(-1, n * 6)):
                res = r - v + t * _reference(xy, rho, table, v.reshape(1, n, 6)).ravel()
                assert np.linalg.norm(res) <= (1e-9 + 1e-12) * np.linalg.norm(r), restart
            assert free_memory() - free < 2 ** 22, restart  # (captured graphs may take some)


def test_threads_solve_while_others_capture(gpu):
    """Each thread solves with operators of its own, one to three right-hand sides, every operator four times: the
    second run of each step captures its graph while the other threads launch on the same stream."""
    from smuthi_amd.linear_system import CouplingMatrixRadialLookupCUDA

    def system(n):
        xy, rho, table = _system(n, n)
        op = CouplingMatrixRadialLookupCUDA.from_table(table, rho, [Sphere([a, b, 200.0], 1.5, 50.0, 1, 1)
                                                                    for a, b in xy], H, 'linear')
        rng = np.random.default_rng(n)
        d = np.hypot(xy[:, None, 0] - xy[None, :, 0], xy[:, None, 1] - xy[None, :, 1])
        t = (0.25 / (6 * (1 / (1 + d / 500)).sum(1).max()) * np.exp(2j * np.pi * rng.uniform(size=(n, 6)))).ravel()
        b = rng.standard_normal((3, n * 6)) + 1j * rng.standard_normal((3, n * 6))
        want = op.solve_master(t, b, 1e-10, precision='double')
        return op, t, b, want

    work = [[system(n) for n in sizes] for sizes in ((20, 90, 41), (33, 60, 25), (70, 28, 52))]
    failures = []

    def solve(systems):
        try:
            for op, t, b, want in systems:
                for repeat in range(4):
                    for rhs, ref in ((b[0], want[0]), (b, want)):
                        for precision in ('double', 'mixed'):
                            x = op.solve_master(t, rhs, 1e-8, precision=precision)
                            err = np.linalg.norm(x - ref) / np.linalg.norm(ref)
                            if not err <= 1e-7:
                                failures.append((op.shape, repeat, precision, err))
        except Exception as e:
            failures.append(e)

    threads = [threading.Thread(target=solve, args=(w,)) for w in work]
    print('solves in %d threads' % len(threads), flush=True)
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures, failures
