"""Batched rSVD at the edges of its row work: 256-row slabs of 64-row chunks, 32-row k blocks of
the passes' tiles, sketch widths from 1 to 48, rows above and below columns.  Against the oracle
with the same Omega, at the batched path's fp32 level (as test_gpu_batched.py)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 31, 33, 48, 64, 65, 255, 256, 257, 320, 511, 513]


@pytest.mark.parametrize("q,p", [(1, 0), (2, 8), (3, 5)])
def test_slab_edges(gpu_lib, oracle, q, p):
    rng = np.random.default_rng(40 + q)
    shapes = [(SIZES[i], SIZES[j]) for i in range(len(SIZES)) for j in range(len(SIZES))
              if min(SIZES[i], SIZES[j]) > p and (i + j) % 3 == q % 3]
    m, n = (np.array(x, dtype=np.int32) for x in zip(*shapes))
    mn = np.minimum(m, n)
    # below full width the residual is the decay's, not rounding: k + p <= mn / 2 where it can be
    k = np.maximum(1, np.minimum(48 - p, mn // 2 - p)).astype(np.int32)
    b = gpu_lib.Batch(m, n, k, p)
    b.fill_test_matrices(rng.uniform(8, 32, len(m)), 17)
    assert b.run(q=q, seed=70) == 0
    for i, (u, s, v) in enumerate(b.results()):
        A = b.matrix(i).astype(np.float64)
        l = int(k[i]) + p
        om = gpu_lib.gaussian(70 + i, 0, int(n[i]) * l).reshape(l, n[i]).T
        Ur, Sr, Vr = oracle.fixed_rank(A, int(k[i]), p, 2, q, 1, omega=om)
        u, v = u.astype(np.float64), v.astype(np.float64)
        assert np.abs(s - np.diag(Sr)).max() < 2e-5, (m[i], n[i], k[i])
        r, rr = np.linalg.norm(A - (u * s) @ v.T), np.linalg.norm(A - Ur @ Sr @ Vr.T)
        assert abs(r - rr) < 1e-3 * rr + 2e-5, (m[i], n[i], k[i], r, rr)
        # Q's last rounding to FP32, 2^-24 of an entry: 2 * 2^-24 an entry of Q^T Q, 48 of them
        # in a sum, and U's own
        assert np.abs(u.T @ u - np.eye(k[i])).max() < 50 * 2.0 ** -23, (m[i], n[i], k[i])
