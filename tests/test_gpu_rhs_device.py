"""The allocation-free RHS on device pointers (two launches): the sums of the
allocating path's GEMV and stage kernels, so the same bits; one block without
couplings, ragged blocks, operators within and past the memory-side cache
(which are read with and without allocating there), and in place."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gauge", ["v", "l"])
@pytest.mark.parametrize("s", [[5], [1, 1], [130, 257, 16, 300],
                               [5700, 5700], [5800, 5800]])
def test_matches_prop_rhs(s, gauge):
    import mpci
    from mpci import _lib, synth
    lib = _lib.tdse_lib()
    hip = C.CDLL("libamdhip64.so.7")
    hip.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
    hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    hip.hipFree.argtypes = [C.c_void_p]
    E, D = synth.system_arrays(s, seed=sum(s))
    g = mpci.System(E, D, gauge=gauge)
    x = np.random.default_rng(1).standard_normal(2 * g.N)
    prop = mpci.Propagator(g)
    prop.set_small_path(0)
    ref = prop.rhs(0.03, x)
    bufs = []
    for host in (x, np.full_like(x, np.nan)):
        p = C.c_void_p()
        assert hip.hipMalloc(C.byref(p), x.nbytes) == 0
        assert hip.hipMemcpy(p, host.ctypes.data, x.nbytes, 1) == 0
        bufs.append(p)
    try:
        for out in (bufs[1], bufs[0]):
            _lib.check(lib.mpci_system_rhs_noalloc(g.h, 0.03, bufs[0], out,
                                                   None))
            got = np.empty_like(x)
            assert hip.hipDeviceSynchronize() == 0
            assert hip.hipMemcpy(got.ctypes.data, out, x.nbytes, 2) == 0
            assert np.array_equal(got, ref)
    finally:
        for p in bufs:
            hip.hipFree(p)
