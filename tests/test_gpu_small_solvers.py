"""The symmetric eigensolver at the sizes where its paths change: one workgroup up to 48, then
blocks of 16 columns in pairs, with padding blocks and columns, against numpy in float64."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = 2.220446049250313e-16


def _psd(n, seed, kind):
    rng = np.random.default_rng(seed)
    Q, _ = np.linalg.qr(rng.standard_normal((n, n)))
    if kind == "decay":
        lam = np.exp(-np.arange(n) * 24.0 / n)
    elif kind == "plateau":
        lam = np.where(np.arange(n) < (n + 1) // 2, 1.0, 1e-9)
    else:
        lam = np.ones(n)
    G = (Q * lam) @ Q.T
    return (G + G.T) / 2


def _eig(rp, G):
    n = G.shape[0]
    d = rp.DeviceMatrix.from_host(G)
    w, V = rp.DeviceMatrix(n, 1), rp.DeviceMatrix(n, n)
    sw = C.c_int(-1)
    rc = rp.load().rsvd_dev_sym_eig_psd(n, d.ptr, n, w.ptr, V.ptr, n, C.byref(sw))
    assert rc == 0, rp.last_error()
    assert 0 <= sw.value < 60
    return w.to_host()[:, 0], V.to_host()


@pytest.mark.parametrize("kind", ["decay", "plateau", "identity"])
@pytest.mark.parametrize("n", [1, 2, 3, 16, 31, 47, 48, 49, 63, 64, 65, 96, 97, 130])
def test_sym_eig_sizes(gpu_lib, n, kind):
    G = _psd(n, n, kind)
    w, V = _eig(gpu_lib, G)
    norm = np.linalg.norm(G, 2)
    # a backward stable solver's error is a modest multiple of n eps ||G||
    tol = 20 * n * EPS
    assert np.max(np.abs(w - np.linalg.eigvalsh(G))) <= tol * norm
    assert np.max(np.abs(V.T @ V - np.eye(n))) <= tol
    assert np.max(np.abs(G @ V - V * w)) <= tol * norm


@pytest.mark.parametrize("scale", [1e-200, 1e-160, 1e140, 1e200])
@pytest.mark.parametrize("n", [20, 70])
def test_sym_eig_scales(gpu_lib, n, scale):
    """Entries whose squares leave the double range: the result is the scaled one."""
    G = _psd(n, 7, "decay")
    w, V = _eig(gpu_lib, G * scale)
    tol = 20 * n * EPS
    assert np.max(np.abs(w / scale - np.linalg.eigvalsh(G))) <= tol
    assert np.max(np.abs(V.T @ V - np.eye(n))) <= tol
