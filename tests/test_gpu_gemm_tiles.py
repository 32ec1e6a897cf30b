"""FP64 / FP32 products at the edges of the GEMM's tiles, of its k blocks (16 FP64, 32 FP32
elements) and of its k slices, every transposition, Grams (A^T A and B B^T, one operand passed
twice), and leading dimensions beyond the rows.  SHAPES and the Grams are cut into 32 x 32 tiles
(a few workgroups); LARGE are the sizes that the cut's model gives 128 x 64 and 64 x 32 tiles."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (31, 33, 15), (32, 32, 16), (33, 31, 17), (127, 64, 31), (128, 65, 32),
          (129, 63, 33), (64, 1, 4097), (1, 64, 700), (400, 26, 200), (257, 300, 1000)]

# (m, n, k) and what the plan cuts it into, with A not transposed where A^T is not named
LARGE = [(945, 1223, 68),     # FP64 128 x 64: a last tile of 49 rows leaves two of its waves idle
         (949, 1242, 68),     # FP64 128 x 64, A^T
         (4247, 34, 1881),    # FP64 128 x 64 in 15 slices: one wave of the last tile has 23 rows
         (4129, 46, 2988),    # FP64 128 x 64, A^T, 15 slices: less than a tile's columns
         (2435, 202, 53),     # FP64 64 x 32: a last tile of 3 rows and 10 columns
         (2843, 176, 49),     # FP64 64 x 32, A^T: 1 of a k block's 16 left over
         (1785, 40, 1669),    # FP64 64 x 32 in 9 slices
         (2253, 41, 1734),    # FP64 64 x 32, A^T, 7 slices
         (2181, 714, 138),    # FP32 128 x 64: a last tile of 5 rows
         (2739, 605, 136),    # FP32 128 x 64, A^T
         (118, 2061, 2388),   # FP32 128 x 64 in 15 slices: less than a tile's rows
         (723, 1125, 99),     # FP32 64 x 32
         (1669, 497, 105),    # FP32 64 x 32, A^T
         (4683, 35, 1775),    # FP32 64 x 32 in 5 slices
         (4571, 41, 1251)]    # FP32 64 x 32, A^T, 5 slices


def _padded(rng, rows, cols, pad, dtype):
    """A (rows + pad) x cols device buffer and the rows x cols matrix in it; the rest is NaN."""
    full = np.full((rows + pad, cols), np.nan, dtype=dtype)
    full[:rows] = rng.standard_normal((rows, cols))
    return full, full[:rows].astype(np.float64)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("ta,tb", [("N", "N"), ("T", "N"), ("N", "T"), ("T", "T")])
def test_gemm_edges(gpu_lib, ta, tb, dtype):
    rp = gpu_lib
    eps = np.finfo(dtype).eps
    for q, (m, n, k) in enumerate(SHAPES):
        rng = np.random.default_rng(100 + q)
        pad = (0, 1, 3)[q % 3]
        fa, A = _padded(rng, *((m, k) if ta == "N" else (k, m)), pad, dtype)
        fb, B = _padded(rng, *((k, n) if tb == "N" else (n, k)), pad, dtype)
        fc, C0 = _padded(rng, m, n, pad, dtype)
        dA, dB, dC = (rp.DeviceMatrix.from_host(x) for x in (fa, fb, fc))
        beta = (0.0, -0.5)[q % 2]
        rc = rp.load().rsvd_dev_gemm(0 if dtype == np.float64 else 1, ta.encode(), tb.encode(), m,
                                     n, k, 2.0, dA.ptr, fa.shape[0], dB.ptr, fb.shape[0], beta,
                                     dC.ptr, fc.shape[0])
        assert rc == 0, rp.last_error()
        oA, oB = (A if ta == "N" else A.T), (B if tb == "N" else B.T)
        got = dC.to_host()
        # every term once: at most k roundings of the running sum, then alpha and beta
        bound = (k + 4) * eps * (2.0 * np.abs(oA) @ np.abs(oB) + np.abs(C0))
        err = np.abs(got[:m] - (2.0 * oA @ oB + beta * C0))
        assert np.all(err <= bound), (m, n, k, float((err / bound).max()))
        assert np.all(np.isnan(got[m:]))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("ta,tb", [("N", "N"), ("T", "N"), ("N", "T"), ("T", "T")])
@pytest.mark.parametrize("m,n,k", LARGE)
def test_larger_tiles(gpu_lib, m, n, k, ta, tb, dtype):
    rp = gpu_lib
    rng = np.random.default_rng(m)
    fa, A = _padded(rng, *((m, k) if ta == "N" else (k, m)), 3, dtype)
    fb, B = _padded(rng, *((k, n) if tb == "N" else (n, k)), 1, dtype)
    fc, C0 = _padded(rng, m, n, 1, dtype)
    dA, dB, dC = (rp.DeviceMatrix.from_host(x) for x in (fa, fb, fc))
    rc = rp.load().rsvd_dev_gemm(0 if dtype == np.float64 else 1, ta.encode(), tb.encode(), m, n, k,
                                 2.0, dA.ptr, fa.shape[0], dB.ptr, fb.shape[0], -0.5, dC.ptr,
                                 fc.shape[0])
    assert rc == 0, rp.last_error()
    oA, oB = (A if ta == "N" else A.T), (B if tb == "N" else B.T)
    got = dC.to_host()
    bound = (k + 4) * np.finfo(dtype).eps * (2.0 * np.abs(oA) @ np.abs(oB) + np.abs(C0))
    err = np.abs(got[:m] - (2.0 * oA @ oB - 0.5 * C0))
    assert np.all(err <= bound), float((err / bound).max())
    assert np.all(np.isnan(got[m:]))


@pytest.mark.parametrize("m,n,kstep", [(1937, 1999, 67), (1300, 331, 20)])
def test_deflation_norm(gpu_lib, m, n, kstep):
    """A <- A - Q B with the sum of squares of the result taken in the same launch, in 128 x 64
    (first size: a last tile of 17 rows and 15 columns, three of its waves idle) and 32 x 32 tiles.
    A tolerance that the first block meets ends the adaptive QB there and returns that norm."""
    rp = gpu_lib
    rng = np.random.default_rng(n)
    A = rng.standard_normal((m, n))
    nstep = -(-min(m, n) // kstep)
    dA = rp.DeviceMatrix.from_host(A)
    dQ, dB = rp.DeviceMatrix(m, kstep * nstep), rp.DeviceMatrix(kstep * nstep, n)
    fr, norm = C.c_int(0), C.c_double(0)
    rc = rp.load().rsvd_dev_randqb(dA.ptr, m, n, m, kstep, 0, 1e9, 0, 1, 1, 5, None, dQ.ptr, m,
                                   dB.ptr, kstep * nstep, C.byref(fr), C.byref(norm))
    assert rc == 0, rp.last_error()
    assert fr.value == kstep
    Q, B = dQ.to_host()[:, :kstep], dB.to_host()[:kstep]
    eps = np.finfo(np.float64).eps
    # an entry's error, here and there, and 4096 roundings in any one chain of the sum of squares
    each = 2.0 * (kstep + 4) * eps * (np.abs(Q) @ np.abs(B) + np.abs(A))
    want = np.linalg.norm(A - Q @ B)
    assert abs(norm.value - want) <= np.linalg.norm(each) + 4096 * eps * want


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n,k", [(1, 5), (20, 2000), (33, 400), (64, 64), (110, 2000),
                                 (129, 5001), (300, 50)])
def test_gram_is_symmetric(gpu_lib, n, k, dtype):
    rp = gpu_lib
    eps = np.finfo(dtype).eps
    rng = np.random.default_rng(n)
    for ta in "TN":
        X = rng.standard_normal((k, n) if ta == "T" else (n, k)).astype(dtype)
        dX, dG = rp.DeviceMatrix.from_host(X), rp.DeviceMatrix(n, n, dtype)
        rc = rp.load().rsvd_dev_gemm(0 if dtype == np.float64 else 1, ta.encode(),
                                     b"N" if ta == "T" else b"T", n, n, k, 1.0, dX.ptr,
                                     X.shape[0], dX.ptr, X.shape[0], 0.0, dG.ptr, n)
        assert rc == 0, rp.last_error()
        G = dG.to_host()
        Y = X.astype(np.float64) if ta == "T" else X.T.astype(np.float64)
        assert np.array_equal(G, G.T)
        assert np.all(np.abs(G - Y.T @ Y) <= (k + 4) * eps * (np.abs(Y).T @ np.abs(Y)))


def test_fp32_sums_stay_short(gpu_lib):
    """An FP32 product with a long k and an output past 2^20 entries: its running sums take at most
    K / 35 = 1728 products.  With positive terms each rounding errs by u / sqrt(3) of the sum so far
    (u = 2^-24): u sqrt(1728) / 3 of a sum, over sqrt(35) independent ones 1.4e-7 in the root mean
    square, and u / sqrt(3) for the last rounding; a single sum a quarter of K long reaches 1.2e-6."""
    rp = gpu_lib
    m = n = 1200
    k = 60000
    rng = np.random.default_rng(4)
    A = rng.uniform(0.5, 1.5, (m, k)).astype(np.float32)
    B = rng.uniform(0.5, 1.5, (k, n)).astype(np.float32)
    dA, dB = rp.DeviceMatrix.from_host(A), rp.DeviceMatrix.from_host(B)
    dC = rp.DeviceMatrix(m, n, np.float32)
    rc = rp.load().rsvd_dev_gemm(1, b"N", b"N", m, n, k, 1.0, dA.ptr, m, dB.ptr, k, 0.0, dC.ptr, m)
    assert rc == 0, rp.last_error()
    want = A.astype(np.float64) @ B.astype(np.float64)
    assert np.sqrt(np.mean((dC.to_host() / want - 1.0) ** 2)) <= 3e-7


@pytest.mark.parametrize("ta,tb", [("N", "N"), ("T", "N"), ("N", "T"), ("T", "T")])
@pytest.mark.parametrize("m,n,k,pad", [(4099, 513, 255, 1), (2561, 1000, 257, 3), (70001, 31, 297, 0),
                                       (9999, 32, 2001, 3), (193, 33, 80011, 1), (97, 200, 30011, 1),
                                       (7777, 900, 41, 0), (1025, 129, 4099, 1)])
def test_fp32_staged_products(gpu_lib, m, n, k, pad, ta, tb):
    """FP32 products of a GFLOP and more: the sizes that stage their operands in LDS (short k, odd
    row-contiguous operands, long k) and, in the other transpositions, those that do not; edges of
    the 128-row and 32 / 64-column tiles, of the 16-deep stages and of the k slices."""
    rp = gpu_lib
    rng = np.random.default_rng(m)
    fa, A = _padded(rng, *((m, k) if ta == "N" else (k, m)), pad, np.float32)
    fb, B = _padded(rng, *((k, n) if tb == "N" else (n, k)), pad, np.float32)
    fc, C0 = _padded(rng, m, n, pad, np.float32)
    dA, dB, dC = (rp.DeviceMatrix.from_host(x) for x in (fa, fb, fc))
    rc = rp.load().rsvd_dev_gemm(1, ta.encode(), tb.encode(), m, n, k, 2.0, dA.ptr, fa.shape[0],
                                 dB.ptr, fb.shape[0], -0.5, dC.ptr, fc.shape[0])
    assert rc == 0, rp.last_error()
    oA, oB = (A if ta == "N" else A.T), (B if tb == "N" else B.T)
    got = dC.to_host()
    bound = (k + 4) * np.finfo(np.float32).eps * (2.0 * np.abs(oA) @ np.abs(oB) + np.abs(C0))
    err = np.abs(got[:m] - (2.0 * oA @ oB - 0.5 * C0))
    assert np.all(err <= bound), float((err / bound).max())
    assert np.all(np.isnan(got[m:]))
