"""bf16 and split-bf16 products on both sides of the small-tile kernel's rule (4 GFLOP; Grams of up
to 1024 columns), and at the edges of its tiles, k blocks (32) and k slices."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (31, 33, 15), (32, 32, 32), (33, 31, 33), (127, 64, 31), (128, 65, 64),
          (129, 63, 65), (64, 1, 4097), (1, 64, 700), (1024, 64, 512), (257, 300, 1000),
          (5003, 101, 31)]


def _bf16(x):
    """x rounded to bf16 (to nearest, ties to even), as float64."""
    b = np.ascontiguousarray(x, np.float32).view(np.uint32).astype(np.uint64)
    b = (b + 0x7FFF + ((b >> 16) & 1)) & 0xFFFF0000
    return b.astype(np.uint32).view(np.float32).astype(np.float64)


def _check(got, A, B, C, split):
    """One unit in the last place of the running FP32 sum a product; a split operand is off by
    2^-18 of itself (its lo plane's rounding) and lo * lo is left out: 3 * 2^-18 < 2^-16."""
    k = A.shape[1]
    if split == 1:
        A, B = _bf16(A), _bf16(B)
    prod = np.abs(A) @ np.abs(B)
    bound = (split * k + 4) * 2.0 ** -23 * (prod + np.abs(C))
    if split == 3:
        bound += 2.0 ** -16 * prod
    err = np.abs(got - (A @ B + C))
    assert np.all(err <= bound), float((err / bound).max())


def _padded(rng, rows, cols, pad):
    full = np.full((rows + pad, cols), np.nan, dtype=np.float32)
    full[:rows] = rng.standard_normal((rows, cols))
    return full


@pytest.mark.parametrize("split", [1, 3])
@pytest.mark.parametrize("ta,tb", [("N", "N"), ("T", "N"), ("N", "T"), ("T", "T")])
def test_edges(gpu_lib, ta, tb, split):
    rp = gpu_lib
    for q, (m, n, k) in enumerate(SHAPES):
        rng = np.random.default_rng(300 + q)
        pad = (0, 1, 4)[q % 3]
        fa = _padded(rng, *((m, k) if ta == "N" else (k, m)), pad)
        fb = _padded(rng, *((k, n) if tb == "N" else (n, k)), pad)
        fc = _padded(rng, m, n, pad)
        dA, dB, dC = (rp.DeviceMatrix.from_host(x) for x in (fa, fb, fc))
        beta = (0.0, -0.5)[q % 2]
        rc = rp.load().rsvd_dev_gemm(2 if split == 1 else 3, ta.encode(), tb.encode(), m, n, k, 2.0,
                                     dA.ptr, fa.shape[0], dB.ptr, fb.shape[0], beta, dC.ptr,
                                     fc.shape[0])
        assert rc == 0, rp.last_error()
        A, B = (x[:x.shape[0] - pad].astype(np.float64) for x in (fa, fb))
        got = dC.to_host()
        assert np.all(np.isnan(got[m:]))
        _check(got[:m], 2.0 * (A if ta == "N" else A.T), B if tb == "N" else B.T,
               beta * fc[:m].astype(np.float64), split)


@pytest.mark.parametrize("split", [1, 3])
@pytest.mark.parametrize("ta,tb", [("N", "N"), ("T", "N"), ("N", "T"), ("T", "T")])
@pytest.mark.parametrize("m,n,k", [(1925, 961, 137), (4489, 323, 144), (559, 910, 2068),
                                   (723, 1125, 99), (1311, 582, 107), (1113, 109, 1770),
                                   (1367, 68, 1775)])
def test_larger_tiles(gpu_lib, m, n, k, ta, tb, split):
    """The sizes that the small-tile kernel's plan cuts into 128 x 64 (the first three, the third
    of them in 6 slices: 5, 9 and 47 rows in the last tile) and 64 x 32 tiles (the last two in 7)."""
    rp = gpu_lib
    rng = np.random.default_rng(m)
    fa = _padded(rng, *((m, k) if ta == "N" else (k, m)), 3)
    fb = _padded(rng, *((k, n) if tb == "N" else (n, k)), 1)
    fc = _padded(rng, m, n, 1)
    dA, dB, dC = (rp.DeviceMatrix.from_host(x) for x in (fa, fb, fc))
    rc = rp.load().rsvd_dev_gemm(2 if split == 1 else 3, ta.encode(), tb.encode(), m, n, k, 2.0,
                                 dA.ptr, fa.shape[0], dB.ptr, fb.shape[0], -0.5, dC.ptr,
                                 fc.shape[0])
    assert rc == 0, rp.last_error()
    A, B = fa[:-3].astype(np.float64), fb[:-1].astype(np.float64)
    got = dC.to_host()
    assert np.all(np.isnan(got[m:]))
    _check(got[:m], 2.0 * (A if ta == "N" else A.T), B if tb == "N" else B.T,
           -0.5 * fc[:m].astype(np.float64), split)


@pytest.mark.parametrize("split", [1, 3])
@pytest.mark.parametrize("n", [1000, 1001])
def test_both_sides_of_the_rule(gpu_lib, n, split):
    rp = gpu_lib
    rng = np.random.default_rng(n)
    A = rng.standard_normal((1000, 2000)).astype(np.float32)
    B = rng.standard_normal((2000, n)).astype(np.float32)
    dA, dB, dC = (rp.DeviceMatrix.from_host(x) for x in (A, B, np.zeros((1000, n), np.float32)))
    rc = rp.load().rsvd_dev_gemm(2 if split == 1 else 3, b"N", b"N", 1000, n, 2000, 1.0, dA.ptr, 1000,
                                 dB.ptr, 2000, 0.0, dC.ptr, 1000)
    assert rc == 0, rp.last_error()
    _check(dC.to_host(), A.astype(np.float64), B.astype(np.float64), np.zeros((1000, n)), split)


@pytest.mark.parametrize("split", [1, 3])
@pytest.mark.parametrize("n,k", [(1, 40), (33, 400), (64, 64), (101, 5003), (129, 4099),
                                 (1024, 70), (1025, 70)])
def test_gram_is_symmetric(gpu_lib, n, k, split):
    rp = gpu_lib
    rng = np.random.default_rng(n)
    X = rng.standard_normal((k, n)).astype(np.float32)
    dX, dG = rp.DeviceMatrix.from_host(X), rp.DeviceMatrix(n, n, np.float32)
    rc = rp.load().rsvd_dev_gemm(2 if split == 1 else 3, b"T", b"N", n, n, k, 1.0, dX.ptr, k, dX.ptr,
                                 k, 0.0, dG.ptr, n)
    assert rc == 0, rp.last_error()
    G = dG.to_host()
    assert np.array_equal(G, G.T)
    _check(G, X.T.astype(np.float64), X.astype(np.float64), np.zeros((n, n)), split)
