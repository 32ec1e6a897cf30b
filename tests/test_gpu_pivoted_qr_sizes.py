"""Column-pivoted QR at the sizes where its step kernel changes: one row or column, columns kept in
registers (512 rows) and beyond, a pivot column that fits its LDS buffer (4096 rows) and one that
does not; ties of the pivot choice.  Pivots and factors against the oracle (dgeqp3 restated)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n", [(1, 1), (1, 6), (6, 1), (3, 64), (64, 300), (300, 65), (513, 40),
                                 (700, 33), (4097, 9), (4500, 5)])
def test_pivoted_qr_sizes(gpu_lib, oracle, m, n):
    rng = np.random.default_rng(m * 31 + n)
    # distinct column scales keep the pivot choices far from ties
    A = rng.standard_normal((m, n)) * np.exp(rng.uniform(-1, 1, n))
    Q, R, I = gpu_lib.pivotedQR_mkl(A)
    Qo, Ro, Io = oracle.pivoted_qr(A)
    assert np.array_equal(I, Io)
    k = min(m, n)
    tol = 50 * 2.2e-16 * np.sqrt(m) * np.linalg.norm(A)
    assert np.abs(R[:k, :n] - Ro[:k, :n]).max() <= tol
    assert np.abs(Q[:, :k].T @ Q[:, :k] - np.eye(k)).max() <= 1e-13
    assert np.linalg.norm(Q[:, :k] @ R[:k, :n] - A[:, I]) <= tol


def test_pivot_ties_take_the_first_place(gpu_lib, oracle):
    """Exactly equal norms (unit columns of one entry each) and a zero matrix: the first place in
    the current order wins, which a swap changes."""
    A = np.zeros((8, 10))
    for j, r in enumerate([3, 1, 4, 0, 5, 7, 2, 6, 3, 1]):
        A[r, j] = 2.0 if j == 4 else 1.0
    for M in (A, np.zeros((5, 7))):
        _, R, I = gpu_lib.pivotedQR_mkl(M)
        _, Ro, Io = oracle.pivoted_qr(M)
        assert np.array_equal(I, Io)
        assert np.allclose(np.abs(R), np.abs(Ro), atol=1e-15)


@pytest.mark.parametrize("m,n", [(40, 3584), (40, 3585), (1, 5000), (3, 9000), (700, 3700),
                                 (8390000, 4)])
def test_pivoted_qr_two_launches_a_step(gpu_lib, oracle, m, n):
    """Both sides of the widest matrix that is factored in one launch a step (3584 columns), wide
    ones, and one of more than 2^25 entries."""
    test_pivoted_qr_sizes(gpu_lib, oracle, m, n)


def test_pivot_ties_in_a_wide_matrix(gpu_lib, oracle):
    """4000 columns of four distinct norms each repeated a thousand times, and a zero matrix."""
    A = np.zeros((6, 4000))
    for j in range(4000):
        A[j % 6, j] = 1.0 + j % 4
    for M in (A, np.zeros((3, 4000))):
        _, R, I = gpu_lib.pivotedQR_mkl(M)
        _, Ro, Io = oracle.pivoted_qr(M)
        assert np.array_equal(I, Io)
        assert np.allclose(np.abs(R), np.abs(Ro), atol=1e-14)


def test_pivoted_qr_time_grows_with_the_columns(gpu_lib):
    """A step's work is a few passes over the matrix: ten times the columns may take ten times as
    long (they take about twice as long, the launches being most of it), not their square."""
    lib = gpu_lib.load()

    def best(m, n):
        A = np.random.default_rng(n).standard_normal((m, n))
        times = []
        try:
            for _ in range(3):
                lib.rsvd_kstats_reset()
                lib.rsvd_kstats_enable(1)
                gpu_lib.pivotedQR_mkl(A)
                times.append(gpu_lib.kstats("pivoted_qr")[0])
        finally:
            lib.rsvd_kstats_enable(0)
            lib.rsvd_kstats_reset()
        return min(times)

    assert best(64, 30000) <= 10.0 * best(64, 3000)
