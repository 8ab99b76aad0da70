"""Callers whose buffers are pinned: uploads and downloads go straight to and from them, as the DMA can,
and not through the library's own pinned memory, which serves pageable buffers; the bytes are the same."""
import ctypes as C
import sys

import numpy as np
import pytest

from morphogenesis_amd import _ffi as F
from tests.test_gpu_transfers import system, words
from tests.test_zz_no_alloc import hip_runtime

pytestmark = pytest.mark.gpu


def bounced(lib):
    n = C.c_uint64()
    assert lib.mg_debug_bounced_copies(C.byref(n)) == F.MG_OK
    return n.value


@pytest.mark.parametrize("n", [262145, 540673])  # FCONC: 16 MB + 64, 33 MB
@pytest.mark.parametrize("offset", [0, 4096 + 64])
def test_pinned_buffers_are_not_copied_twice(built, n, offset):
    print("case: pinned buffers,", n * 64, "bytes at", offset, flush=True)
    sys.stdout.flush()
    hip = hip_runtime()
    hip.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
    hip.hipHostFree.argtypes = [C.c_void_p]
    sim = system(n)
    lib, size = sim.lib, n * F.NUM_TF * 4
    p = C.c_void_p()
    assert hip.hipHostMalloc(C.byref(p), size + offset, 0) == 0
    at = C.c_void_p(p.value + offset)
    pinned = np.frombuffer((C.c_char * size).from_address(at.value), np.float32)
    plain = np.empty(size // 4, np.float32)
    try:
        want = words(np.random.default_rng(n), (size // 4,), np.float32)
        pinned[:] = want
        before = bounced(lib)
        assert lib.mg_upload(sim.h, F.FCONC, at, size) == F.MG_OK
        pinned[:] = 0
        assert lib.mg_download(sim.h, F.FCONC, at, size) == F.MG_OK
        assert np.array_equal(pinned.view(np.uint32), want.view(np.uint32))
        assert bounced(lib) == before
        # a pageable buffer in the same process still takes the pinned halves
        assert lib.mg_download(sim.h, F.FCONC, plain.ctypes.data_as(C.c_void_p), size) == F.MG_OK
        assert np.array_equal(plain.view(np.uint32), want.view(np.uint32))
        assert bounced(lib) == before + 1
    finally:
        sim.close()
        hip.hipHostFree(p)


def test_threads_each_with_a_handle(built):
    """Large copies of several handles from several threads at once; a thread's failure is the test's."""
    from concurrent.futures import ThreadPoolExecutor

    def work(k):
        rng = np.random.default_rng(k)
        sim = system(263000 + 777 * k)
        for _ in range(4):
            conc = words(rng, (sim.n, F.NUM_TF), np.float32)
            sim.upload(F.FCONC, conc)
            assert np.array_equal(sim.download(F.FCONC).view(np.uint32), conc.view(np.uint32)), k
        sim.close()
        return k

    print("case: five threads, a handle each", flush=True)
    with ThreadPoolExecutor(5) as pool:
        assert [f.result() for f in [pool.submit(work, k) for k in range(5)]] == list(range(5))
