"""Kernels at the sizes where their loops and dispatch rules change over:
remainders of unrolled loads, edges of tiles, the smallest and largest of a
rule's range, against the oracle or a plain sum."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip(ccnm):
    ccnm.lib()   # the library loads the image's HIP runtime; the test uses the same one
    rt = C.CDLL("libamdhip64.so.7")
    rt.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
    rt.hipFree.argtypes = [C.c_void_p]
    rt.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    rt.hipDeviceSynchronize.argtypes = []
    return rt


@pytest.mark.parametrize("n", [0, 1, 255, 2047, 2048, 2049, 4096 * 2048, 4096 * 2048 + 1, 4097 * 2048 + 300])
def test_energy_noalloc_sum_at_span_edges(ccnm, hip, n):
    """Spans of 2048 amplitudes up to 4096 partials, then longer ones.  A
    thread adds at most 16 products in a row here (longer spans: 2 x 8), the
    trees above it 6 + 4 + 4 + 6 + 16 more, each rounding by at most 2^-53 of
    the sum of moduli, and a product by 2^-52: 64 * 2^-53 covers them."""
    rng = np.random.default_rng(n)
    t, r0 = (rng.standard_normal(2 * n).view(np.complex128) for _ in range(2))
    dev = []
    try:
        for a in (t, r0, np.full(1, 7.0 + 7.0j)):
            p = C.c_void_p()
            assert hip.hipMalloc(C.byref(p), max(a.nbytes, 16)) == 0
            dev.append(p)
            if a.nbytes:
                assert hip.hipMemcpy(p, a.ctypes.data, a.nbytes, 1) == 0
        out = np.zeros(1, np.complex128)
        for _ in range(2):
            ccnm.energy_noalloc(n, dev[0].value, dev[1].value, dev[2].value, None)
            assert hip.hipDeviceSynchronize() == 0
            assert hip.hipMemcpy(out.ctypes.data, dev[2], 16, 2) == 0
    finally:
        for p in dev:
            hip.hipFree(p)
    prod = t * np.conj(r0)
    want = complex(np.sum(prod.real.astype(np.longdouble)), np.sum(prod.imag.astype(np.longdouble)))
    assert abs(out[0] - want) <= 64 * 2.0 ** -53 * np.sum(np.abs(t) * np.abs(r0))
