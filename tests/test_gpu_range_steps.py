"""The fixed-rank SVD's orthonormalisation steps where one Cholesky factor is enough, where the
second one is needed and where the factorisation breaks down, against the oracle on the same
Omega (vnum = 1: the small SVD keeps small singular values)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SPECTRA = {"mild": lambda j: np.exp(-j / 20.0),
           "steep": lambda j: 10.0 ** (-j / 6.0),          # cond(Y) about 3e5 at 33 columns
           "breakdown": lambda j: 10.0 ** (-j / 2.0),      # 1e16: past the pivot test
           "rank 12": lambda j: np.where(j < 12, 1.0 / (1.0 + j), 0.0)}


@pytest.mark.parametrize("spectrum", SPECTRA)
@pytest.mark.parametrize("q,s", [(1, 1), (2, 1), (3, 1), (3, 2)])
def test_against_oracle(gpu_lib, oracle, spectrum, q, s):
    m, n, k, p = 257, 130, 26, 7
    rng = np.random.default_rng(3)
    sigma = SPECTRA[spectrum](np.arange(float(n)))
    U0, V0 = (np.linalg.qr(rng.standard_normal((d, n)))[0] for d in (m, n))
    A = (U0 * sigma) @ V0.T
    gpu_lib.set_seed(99)
    try:
        U, S, V = gpu_lib.low_rank_svd_rand_decomp_fixed_rank(A, k, p, 1, q, s)
    finally:
        gpu_lib.use_time_seed()
    Ur, Sr, Vr = oracle.fixed_rank(A, k, p, 1, q, s, seed=99)
    # the suite's bound for FP64 parity, of sigma_0 = 1
    assert np.abs(np.diag(S) - np.diag(Sr)).max() < 1e-10
    assert abs(np.linalg.norm(A - U @ S @ V.T) - np.linalg.norm(A - Ur @ Sr @ Vr.T)) < 1e-10
    # columns whose own rounding, eps / sigma_j, is below 1e-9
    keep = np.diag(S) > 1e-6
    for X in (U[:, keep], V[:, keep]):
        assert np.abs(X.T @ X - np.eye(keep.sum())).max() < 1e-9


def test_breakdown_leaves_nothing_behind(gpu_lib):
    """A call whose orthonormalisations all break down (a zero matrix) between two calls on a
    full-rank matrix: the second of them queues the products the first did, so no Cholesky
    verdict of the call in between is read again."""
    rp = gpu_lib
    lib = rp.load()
    m, n, k = 300, 200, 24
    A = np.random.default_rng(8).standard_normal((m, n))
    dA = rp.DeviceMatrix.from_host(A)
    dZ = rp.DeviceMatrix.from_host(np.zeros((m, n)))
    U, S, V = rp.DeviceMatrix(m, k), rp.DeviceMatrix(k, 1), rp.DeviceMatrix(n, k)

    def call(X):
        rc = lib.rsvd_dev_fixed_rank(X.ptr, m, n, m, k, 6, 1, 2, 1, 5, None, U.ptr, m, S.ptr,
                                     V.ptr, n)
        assert rc == 0, rp.last_error()
        return rp.kstats("gemm_f64")[1], S.to_host()

    lib.rsvd_kstats_reset()
    lib.rsvd_kstats_enable(1)
    try:
        c0, s0 = call(dA)
        c1, s1 = call(dZ)
        c2, s2 = call(dA)
    finally:
        lib.rsvd_kstats_enable(0)
        lib.rsvd_kstats_reset()
    assert c1 - c0 != c0 and c2 - c1 == c0
    assert np.all(s1 == 0.0) and np.array_equal(s0, s2)


@pytest.mark.parametrize("rank,factors", [(60, 2), (12, 1)])
def test_one_qr_after_a_breakdown(gpu_lib, rank, factors):
    """The last orthonormalisation (q = 1: the only one) factors two Grams, or one that breaks
    down: the Householder QR that follows is the end of it."""
    rp = gpu_lib
    lib = rp.load()
    m, n, k = 300, 200, 24
    rng = np.random.default_rng(9)
    dA = rp.DeviceMatrix.from_host(rng.standard_normal((m, rank)) @ rng.standard_normal((rank, n)))
    U, S, V = rp.DeviceMatrix(m, k), rp.DeviceMatrix(k, 1), rp.DeviceMatrix(n, k)
    lib.rsvd_kstats_reset()
    lib.rsvd_kstats_enable(1)
    try:
        rc = lib.rsvd_dev_fixed_rank(dA.ptr, m, n, m, k, 6, 2, 1, 1, 5, None, U.ptr, m, S.ptr,
                                     V.ptr, n)
        assert rc == 0, rp.last_error()
        count = rp.kstats("chol_inv")[1]
    finally:
        lib.rsvd_kstats_enable(0)
        lib.rsvd_kstats_reset()
    assert count == factors
