"""rsvd_dev_fixed_rank_noalloc near its scratch limit: panels of 180 to 250 MiB, so that little is
left for the products' k slices.  Every shape is one whose panels and factors fit; each against
rsvd_dev_fixed_rank on the same matrix and Omega (a Gaussian A: singular values of one order, the
two differ by the rounding of differently sliced sums)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k,p,vnum,q,s,omega", [
    (2628, 6725, 1013, 10, 2, 2, 2, False),   # B B^T and the QR's Grams
    (8303, 4466, 990, 10, 2, 2, 2, True),
    (6664, 5118, 864, 10, 2, 2, 1, False),
    (12000, 9000, 500, 10, 1, 2, 1, False),   # a product of a whole panel
    (22344, 23872, 237, 10, 1, 2, 1, False),  # n > m: panels that must not move
])
def test_noalloc_near_the_scratch_limit(gpu_lib, m, n, k, p, vnum, q, s, omega):
    rp = gpu_lib
    lib = rp.load()
    dA, dO = rp.DeviceMatrix(m, n), rp.DeviceMatrix(n, k + p) if omega else None
    assert lib.rsvd_dev_gaussian(5, m, n, dA.ptr, m) == 0
    if omega:
        assert lib.rsvd_dev_gaussian(6, n, k + p, dO.ptr, n) == 0
    out = []
    for fn in (lib.rsvd_dev_fixed_rank, lib.rsvd_dev_fixed_rank_noalloc):
        U, S, V = rp.DeviceMatrix(m, k), rp.DeviceMatrix(k, 1), rp.DeviceMatrix(n, k)
        rc = fn(dA.ptr, m, n, m, k, p, vnum, q, s, 7, dO.ptr if omega else None, U.ptr, m, S.ptr,
                V.ptr, n)
        assert rc == 0, rp.last_error()
        out.append((S.to_host()[:, 0], U.to_host()))
    (s0, _), (s1, U) = out
    np.testing.assert_allclose(s1, s0, rtol=1e-11)
    assert np.abs(U.T @ U - np.eye(k)).max() <= 1e-11
