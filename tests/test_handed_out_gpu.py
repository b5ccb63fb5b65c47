"""A handle whose address was handed out ends only when work on other streams is
done with its state, although a later handle may take its memory at once."""
import ctypes as C

import numpy as np
import pytest

from tests.test_zz_no_alloc import _hip

pytestmark = pytest.mark.gpu


def test_close_while_another_stream_reads():
    from qiskit_aer_amd import QubitVector
    print("case: close while another stream reads", flush=True)
    n = 22
    size = 16 << n
    hip = _hip()
    hip.hipMemcpyAsync.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int, C.c_void_p]
    hip.hipStreamCreate.argtypes = [C.POINTER(C.c_void_p)]
    hip.hipStreamSynchronize.argtypes = hip.hipStreamDestroy.argtypes = [C.c_void_p]
    out, side = C.c_void_p(), C.c_void_p()
    e = QubitVector(n)
    assert hip.hipMalloc(C.byref(out), size) == 0 and hip.hipStreamCreate(C.byref(side)) == 0
    try:
        e.initialize_random(5)
        want = e.copy_to_vector()
        ptr = e.device_pointer()
        for _ in range(100):  # some milliseconds of reads (3: device to device)
            assert hip.hipMemcpyAsync(out, ptr, size, 3, side) == 0
        e.close()
        later = QubitVector(n)  # of the same size: takes the memory
        later.initialize()
        later.synchronize()
        assert hip.hipStreamSynchronize(side) == 0
        got = np.empty(1 << n, dtype=np.complex128)
        assert hip.hipMemcpy(got.ctypes.data, out, size, 2) == 0
        assert np.array_equal(got, want)
        later.close()
    finally:
        assert hip.hipDeviceSynchronize() == 0
        hip.hipStreamDestroy(side)
        hip.hipFree(out)
