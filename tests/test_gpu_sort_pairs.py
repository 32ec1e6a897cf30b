"""The order of eigenpairs on either side of a wave of 64 values: a diagonal matrix, which the
solver leaves as it is, with ties, which keep their order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 5, 63, 64, 65, 129, 300])
def test_ties_keep_their_order(gpu_lib, n):
    rp = gpu_lib
    d = np.random.default_rng(n).integers(1, max(3, n // 3), n).astype(np.float64)
    dG = rp.DeviceMatrix.from_host(np.diag(d))
    dV, dl = rp.DeviceMatrix(n, n), rp.DeviceMatrix(n, 1)
    rc = rp.load().rsvd_dev_sym_eig_psd(n, dG.ptr, n, dl.ptr, dV.ptr, n, None)
    assert rc == 0, rp.last_error()
    order = np.argsort(d, kind="stable")
    assert np.array_equal(dl.to_host()[:, 0], d[order])
    assert np.array_equal(dV.to_host(), np.eye(n)[:, order])
