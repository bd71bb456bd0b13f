"""Direct field sums whose particles are split over workgroups: one particle and
one point, a whole chunk of 32 and one more, many particles at few points, several
chunks in one workgroup, for
the unrolled kernels (m_max = l_max, below it, 4) and the runtime-order one,
E and H, against the oracle's sum. FP64: the recurrences and sums keep a few
1e-16 per term, 1e-11 as the kernel's own test; FP32: a few roundings of 6e-8
per recurrence step at k r > 1, 2e-5 as that test."""
import numpy as np
import pytest

from oracle import swe as osw

pytestmark = pytest.mark.gpu

K = 2 * np.pi / 550


@pytest.fixture(scope='module')
def gpu():
    from smuthi_amd import cuda
    assert cuda.enable_gpu(), 'MI355X not available'
    return cuda


@pytest.mark.parametrize('l_max,m_max', [(1, 1), (3, 3), (3, 2), (4, 4), (5, 3)])
@pytest.mark.parametrize('n,points', [(1, 1), (32, 300), (33, 257), (150, 5)])
def test_split_sums_match_oracle(gpu, n, points, l_max, m_max):
    from smuthi_amd import fields
    from smuthi_amd.expansions import swe_field_sum
    rng = np.random.default_rng(n + points + l_max)
    B = fields.blocksize(l_max, m_max)
    pos = np.stack([rng.uniform(-3000, 3000, n), rng.uniform(-3000, 3000, n), rng.uniform(100, 300, n)], 1)
    pts = np.stack([rng.uniform(-3000, 3000, points), rng.uniform(-3000, 3000, points),
                    rng.uniform(420, 2000, points)], 1)
    pts[0, :2] = pos[0, :2]  # on a particle's axis
    coef = rng.standard_normal((n, B)) + 1j * rng.standard_normal((n, B))
    k = K * (1 + 0.02j) if l_max == 3 else K
    print('swe splits: %d particles, %d points, l_max %d' % (n, points, l_max), flush=True)
    for field in ('E', 'H'):
        want = np.stack(osw.direct_field([(c, l_max, m_max, p, 90.0) for c, p in zip(coef, pos)], k, *pts.T,
                                         field=field, omega=K))
        for precision, tol in (('double', 1e-11), ('single', 2e-5)):
            got = np.stack(swe_field_sum(pos, np.full(n, 90.0), np.tile([-np.inf, np.inf], (n, 1)), coef, l_max, m_max,
                                         k, pts, 0 if field == 'E' else 1, K, precision))
            assert np.linalg.norm(got - want) <= tol * np.linalg.norm(want), (field, precision)


@pytest.mark.parametrize('l_max,m_max', [(3, 3), (5, 3)])
def test_workgroups_of_several_chunks(gpu, l_max, m_max):
    """So many points that a workgroup takes more than a chunk of 32 particles: 700 in eight splits, of two chunks and
    24 more (the last one 20); a few of the points are checked."""
    from smuthi_amd import fields
    from smuthi_amd.expansions import swe_field_sum
    rng = np.random.default_rng(l_max)
    n, points = 700, 70000
    B = fields.blocksize(l_max, m_max)
    pos = np.stack([rng.uniform(-3000, 3000, n), rng.uniform(-3000, 3000, n), rng.uniform(100, 300, n)], 1)
    pts = np.stack([rng.uniform(-3000, 3000, points), rng.uniform(-3000, 3000, points),
                    rng.uniform(420, 2000, points)], 1)
    coef = rng.standard_normal((n, B)) + 1j * rng.standard_normal((n, B))
    some = np.array([0, 255, 256, 30000, 69887, 69888, 69999])
    print('swe chunks: %d particles, %d points, l_max %d' % (n, points, l_max), flush=True)
    want = np.stack(osw.direct_field([(c, l_max, m_max, p, 90.0) for c, p in zip(coef, pos)], K, *pts[some].T,
                                     field='E', omega=K))
    for precision, tol in (('double', 1e-11), ('single', 2e-5)):
        got = np.stack(swe_field_sum(pos, np.full(n, 90.0), np.tile([-np.inf, np.inf], (n, 1)), coef, l_max, m_max, K,
                                     pts, 0, K, precision))[:, some]
        assert np.linalg.norm(got - want) <= tol * np.linalg.norm(want), precision
