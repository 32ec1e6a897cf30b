"""The k slices of a product of large dimensions: the device memory that the library takes for
them is bounded (2^28 elements), whatever the size of the output."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_slices_of_a_large_output(gpu_lib):
    rp = gpu_lib
    lib = rp.load()
    hip = C.CDLL("libamdhip64.so")
    hip.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t), C.POINTER(C.c_size_t)]

    def free_mem():
        free, total = C.c_size_t(0), C.c_size_t(0)
        assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    m, n, k = 13593, 8853, 45164
    dA, dB, dC = (rp.DeviceMatrix(r, c, np.float32) for r, c in ((m, k), (k, n), (m, n)))
    for d in (dA, dB):
        assert lib.rsvd_memset_dev(d.ptr, 0, d.nbytes) == 0
    lib.rsvd_release_cache()
    free0 = free_mem()
    rc = lib.rsvd_dev_gemm(1, b"N", b"N", m, n, k, 1.0, dA.ptr, m, dB.ptr, k, 0.0, dC.ptr, m)
    assert rc == 0, rp.last_error()
    taken = free0 - free_mem()
    lib.rsvd_release_cache()
    assert taken <= 4 * 2 ** 28 + (64 << 20), taken
