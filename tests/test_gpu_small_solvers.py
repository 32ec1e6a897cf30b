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


@pytest.mark.parametrize("n,rank", [(64, 64), (65, 30), (200, 1), (1000, 64)])
def test_sketch_features_of_64_rows(gpu_lib, n, rank):
    """The eigenvalue-only solver behind the features.  With m = 64 rows the sketch's basis Q is
    square, so the features are those of A itself whatever the sketch's rounding."""
    rp = gpu_lib
    m = 64
    rng = np.random.default_rng(n)
    A = rng.standard_normal((m, rank)) @ np.diag(np.exp(-np.arange(rank) / 6.0)) \
        @ rng.standard_normal((rank, n))
    A32 = (A + 1e-3 * rng.standard_normal((m, n))).astype(np.float32)
    A = A32.astype(np.float64)
    d64, d32 = rp.DeviceMatrix.from_host(A), rp.DeviceMatrix.from_host(A32)
    f = rp.DeviceMatrix(64, 1, np.float32)
    rp._check(rp.load().rsvd_dev_sketch_features(d64.ptr, d32.ptr, m, n, m, 5, f.ptr))
    s = np.linalg.svd(A, compute_uv=False)
    a2 = np.sum(A * A)
    t = np.maximum(a2 - np.cumsum(s ** 2), 1e-16 * a2) / a2
    # an absolute error of about 64 eps in t: 1e-4 of t at 1e-10, 5e-6 of its logarithm / 8
    ok = t > 1e-10
    assert ok.sum() >= 20
    assert np.max(np.abs(f.to_host()[ok, 0] - np.log10(t[ok]) / 8)) <= 1e-5


@pytest.mark.parametrize("B", [1, 16, 1024, 1025])
def test_mlp_forward_batches(gpu_lib, B):
    """Both forward kernels (one sample a workgroup, sixteen) against float64."""
    from oracle import mlp
    rp = gpu_lib
    rng = np.random.default_rng(B)
    th = (mlp.init_params(9) + 0.05 * rng.standard_normal(mlp.n_params())).astype(np.float32)
    X = rng.standard_normal((B, 64)).astype(np.float32)
    dth = rp.DeviceMatrix.from_host(th.reshape(-1, 1))
    dX = rp.DeviceMatrix.from_host(X.reshape(-1, 1))
    dO = rp.DeviceMatrix(B * 6, 1, np.float32)
    rp._check(rp.load().rsvd_dev_mlp_forward(dth.ptr, dX.ptr, B, dO.ptr))
    want, _ = mlp.forward(th.astype(np.float64), X.astype(np.float64))
    # four layers of 128-term float sums
    tol = 4 * 128 * 2.0 ** -24
    assert np.abs(dO.to_host().reshape(B, 6) - want).max() <= tol * (1 + np.abs(want).max())
