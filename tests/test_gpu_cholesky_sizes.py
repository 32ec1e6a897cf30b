"""CholeskyQR2 at the edges of its 16-column blocks and 32-column panels: Q orthonormal, Q R = M,
R upper triangular with a positive diagonal, and the pivot test's fallback in each block."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 64, 65, 96, 100]


@pytest.mark.parametrize("n", SIZES)
def test_qr_block_edges(gpu_lib, n):
    rng = np.random.default_rng(n)
    m = n + 37
    M = rng.standard_normal((m, n)) * np.logspace(0, -2, n)
    Q, R = gpu_lib.compact_QR_factorization(M)
    # two Cholesky passes leave a few n eps
    tol = 10 * (n + 16) * 2.2e-16
    assert np.abs(Q.T @ Q - np.eye(n)).max() <= tol
    assert np.array_equal(np.tril(R, -1), np.zeros((n, n)))
    assert np.all(np.diag(R) > 0)
    assert np.linalg.norm(Q @ R - M) <= tol * np.linalg.norm(M) * np.sqrt(n)


@pytest.mark.parametrize("n,j", [(17, 16), (33, 15), (33, 32), (64, 40), (70, 69)])
def test_dependent_column_takes_the_fallback(gpu_lib, n, j):
    rng = np.random.default_rng(n + j)
    M = rng.standard_normal((200, n))
    M[:, j] = M[:, 0] - 2.0 * M[:, j - 1]
    Q = gpu_lib.QR_factorization_getQ(M)
    assert np.abs(Q.T @ Q - np.eye(n)).max() <= 1e-13
    assert np.linalg.norm(Q @ (Q.T @ M) - M) <= 1e-12 * np.linalg.norm(M)
