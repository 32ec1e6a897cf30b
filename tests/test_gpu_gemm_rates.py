"""Rates of products at odd sizes, whose matrix rows straddle cache lines; the fastest of ten calls."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rate(rp, tag, dtype, ta, tb, m, n, k):
    lib = rp.load()
    ar, ac = (m, k) if ta == b"N" else (k, m)
    br, bc = (k, n) if tb == b"N" else (n, k)
    rng = np.random.default_rng(1)
    dA = rp.DeviceMatrix.from_host(rng.random((ar, ac), dtype=dtype))
    dB, dC = rp.DeviceMatrix.from_host(rng.random((br, bc), dtype=dtype)), rp.DeviceMatrix(m, n, dtype)
    best = np.inf
    try:
        for _ in range(10):
            lib.rsvd_kstats_reset()
            lib.rsvd_kstats_enable(1)
            rc = lib.rsvd_dev_gemm(0 if dtype == np.float64 else 1, ta, tb, m, n, k, 1.0, dA.ptr, ar,
                                   dB.ptr, br, 0.0, dC.ptr, m)
            assert rc == 0, rp.last_error()
            best = min(best, rp.kstats(tag)[0])
    finally:
        lib.rsvd_kstats_enable(0)
        lib.rsvd_kstats_reset()
    return 2e-9 * m * n * k / best


@pytest.mark.parametrize("m,n,k,least", [(4013, 50, 18712, 27.0), (2271, 110, 14730, 30.0),
                                         (100, 4073, 43721, 29.0)])
def test_transposed_product_rate(gpu_lib, m, n, k, least):
    """FP64 A^T B with a narrow output: a cut into one long workgroup a CU waits for its operands (20
    to 26 TFLOP/s); the present ones reach 32 to 36."""
    assert _rate(gpu_lib, "gemm_f64", np.float64, b"T", b"N", m, n, k) >= least


@pytest.mark.parametrize("m,n,k,least", [(4987, 576, 18539, 49.0), (36655, 384, 3765, 51.0)])
def test_large_transposed_product_rate(gpu_lib, m, n, k, least):
    """FP64 A^T B past 40 GFLOP with a tall output: 32 x 32 tiles reach 40 and 47 TFLOP/s (their
    reads take all that the memory gives), 64 x 32 ones 57 and 58."""
    assert _rate(gpu_lib, "gemm_f64", np.float64, b"T", b"N", m, n, k) >= least


@pytest.mark.parametrize("m,n,k,least", [(4909, 1389, 18210, 84.0), (41572, 294, 9769, 75.0)])
def test_large_transposed_product_rate_fp32(gpu_lib, m, n, k, least):
    """FP32 A^T B past 20 GFLOP: 72 and 66 TFLOP/s with 32 x 32 tiles, 97 and 85 with larger ones."""
    assert _rate(gpu_lib, "gemm_f32", np.float32, b"T", b"N", m, n, k) >= least


@pytest.mark.parametrize("m,n,k", [(50001, 301, 3005), (5001, 2003, 1005)])
def test_fp32_row_contiguous_rate(gpu_lib, m, n, k):
    """FP32 A B^T: staged operands reach 80 TFLOP/s and more, fed to registers by each wave 46."""
    assert _rate(gpu_lib, "gemm_f32", np.float32, b"N", b"T", m, n, k) >= 62.0


@pytest.mark.parametrize("n,k,least", [(640, 65536, 340.0), (512, 131072, 270.0)])
def test_split_bf16_gram_of_whole_tiles(gpu_lib, n, k, least):
    """A long split-bf16 Gram whose columns fill the 128-column staged tiles, in TFLOP/s of the full
    product: 435 and 297 there, 252 and 243 with operands that each wave fetches for itself."""
    rp = gpu_lib
    lib = rp.load()
    A = np.random.default_rng(1).standard_normal((k, n), dtype=np.float32)
    dA, dG = rp.DeviceMatrix.from_host(A), rp.DeviceMatrix(n, n, np.float32)
    best = np.inf
    try:
        for _ in range(10):
            lib.rsvd_kstats_reset()
            lib.rsvd_kstats_enable(1)
            rc = lib.rsvd_dev_gemm(3, b"T", b"N", n, n, k, 1.0, dA.ptr, k, dA.ptr, k, 0.0, dG.ptr, n)
            assert rc == 0, rp.last_error()
            best = min(best, rp.kstats("gemm_bf16")[0])
    finally:
        lib.rsvd_kstats_enable(0)
        lib.rsvd_kstats_reset()
    assert 2e-9 * n * n * k / best >= least
