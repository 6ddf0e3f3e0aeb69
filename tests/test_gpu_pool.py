"""Freed blocks kept by the library: handed out again on the stream that
freed them and on no other, bounded, given back on request and with their
stream, and not for streams that the library did not create."""

import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MIB = 1 << 20
_vp = ctypes.c_void_p


@pytest.fixture
def lib(wb):
    L = wb.lib()
    wb.sync()
    L.wbfmm_hip_pool_release()
    assert L.wbfmm_hip_pool_bytes() == 0
    yield L
    L.wbfmm_hip_set_stream(None, None)
    wb.sync()
    L.wbfmm_hip_pool_release()


def take(L, n):
    p = _vp()
    assert L.wbfmm_hip_malloc(ctypes.byref(p), n) == 0
    return p.value


def test_reused_on_its_stream_only(wb, lib):
    a = take(lib, 3 * MIB)
    lib.wbfmm_hip_free(a)
    assert lib.wbfmm_hip_pool_bytes() == 3 * MIB
    s = _vp()
    assert lib.wbfmm_hip_stream_create(ctypes.byref(s)) == 0
    lib.wbfmm_hip_set_stream(s, None)
    b = take(lib, 3 * MIB)
    assert b != a and lib.wbfmm_hip_pool_bytes() == 3 * MIB
    lib.wbfmm_hip_free(b)
    assert lib.wbfmm_hip_pool_bytes() == 6 * MIB
    lib.wbfmm_hip_set_stream(None, None)
    assert lib.wbfmm_hip_stream_destroy(s) == 0        # b's block goes with its stream
    assert lib.wbfmm_hip_pool_bytes() == 3 * MIB
    assert take(lib, 3 * MIB - 100) == a               # a little smaller: the same block
    assert lib.wbfmm_hip_pool_bytes() == 0
    lib.wbfmm_hip_free(a)
    c = take(lib, MIB)                                 # much smaller: not that block
    assert c != a and lib.wbfmm_hip_pool_bytes() == 3 * MIB
    lib.wbfmm_hip_free(c)


def test_bounded(wb, lib):
    ps = [take(lib, 200 * MIB) for _ in range(8)] + [take(lib, 300 * MIB)]
    for p in ps:
        lib.wbfmm_hip_free(p)
    assert 0 < lib.wbfmm_hip_pool_bytes() <= 1024 * MIB
    assert lib.wbfmm_hip_pool_bytes() % (200 * MIB) == 0   # (300 MiB: never kept)
    assert lib.wbfmm_hip_pool_release() == 0 and lib.wbfmm_hip_pool_bytes() == 0


def test_bounded_in_number(wb, lib):
    """however small they are, at most 16384 blocks are kept, the last freed"""
    ps = [take(lib, 4096) for _ in range(20000)]
    for p in ps:
        lib.wbfmm_hip_free(p)
    assert lib.wbfmm_hip_pool_bytes() == 16384 * 4096
    a = take(lib, 4096)
    assert a in ps[-16384:]
    lib.wbfmm_hip_free(a)


def test_smallest_that_fits(wb, lib):
    """of the kept blocks the smallest that holds the request, no more than a
    quarter and a page larger, whatever the order they were freed in"""
    sizes = [40, 10, 24, 12, 30, 11]
    ps = {m: take(lib, m * MIB) for m in sizes}
    for p in ps.values():
        lib.wbfmm_hip_free(p)
    for want, got in ((11, 11), (11, 12), (20, 24), (25, 30), (35, 40), (9, 10)):
        assert take(lib, want * MIB) == ps[got]
    assert lib.wbfmm_hip_pool_bytes() == 0
    for p in ps.values():
        lib.wbfmm_hip_free(p)
    a = take(lib, 15 * MIB)                                # 24 is too large
    assert a not in ps.values()
    lib.wbfmm_hip_free(a)


def runtime():
    """the HIP runtime that the library has loaded"""
    path = next(l.split()[-1] for l in open("/proc/self/maps") if "libamdhip64" in l)
    return ctypes.CDLL(path)


@pytest.mark.parametrize("mib", [2, 300])               # below and above the largest kept block
@pytest.mark.parametrize("foreign", [False, True])      # on the library's stream, on a caller's
def test_given_back_when_the_runtime_is_out_of_memory(wb, lib, mib, foreign):
    """an allocation that the runtime refuses is tried again after the kept
    blocks of every stream are given back, whatever its size and stream; with
    nothing to give back it fails"""
    hip = runtime()
    own, s = _vp(), _vp()
    assert lib.wbfmm_hip_stream_create(ctypes.byref(own)) == 0
    for st in (None, own):
        lib.wbfmm_hip_set_stream(st, None)
        lib.wbfmm_hip_free(take(lib, 40 * MIB))
    lib.wbfmm_hip_set_stream(None, None)
    assert lib.wbfmm_hip_pool_bytes() == 80 * MIB
    assert hip.hipStreamCreate(ctypes.byref(s)) == 0
    lib.wbfmm_hip_set_stream(s if foreign else None, None)
    lib.wbfmm_hip_debug_fail_mallocs(1)
    a = take(lib, mib * MIB)
    assert lib.wbfmm_hip_pool_bytes() == 0
    lib.wbfmm_hip_debug_fail_mallocs(1)
    p = _vp()
    assert lib.wbfmm_hip_malloc(ctypes.byref(p), mib * MIB) != 0 and not p.value
    lib.wbfmm_hip_debug_fail_mallocs(0)
    assert lib.wbfmm_hip_malloc(ctypes.byref(p), mib * MIB) == 0
    lib.wbfmm_hip_free(p)
    lib.wbfmm_hip_free(a)
    lib.wbfmm_hip_set_stream(None, None)
    assert hip.hipStreamSynchronize(s) == 0 and hip.hipStreamDestroy(s) == 0
    assert lib.wbfmm_hip_stream_destroy(own) == 0


def test_blocks_of_a_capturing_stream_stay(wb, lib):
    """while a stream is captured its kept blocks are neither released nor
    evicted: the graph has no node for them, and they are released afterwards"""
    hip = runtime()
    s, g, nodes = _vp(), _vp(), ctypes.c_size_t(99)
    assert lib.wbfmm_hip_stream_create(ctypes.byref(s)) == 0
    lib.wbfmm_hip_set_stream(s, None)
    lib.wbfmm_hip_free(take(lib, 100 * MIB))
    lib.wbfmm_hip_set_stream(None, None)
    ps = [take(lib, 200 * MIB) for _ in range(5)]
    assert hip.hipStreamBeginCapture(s, 2) == 0            # relaxed mode
    assert lib.wbfmm_hip_pool_release() == 0 and lib.wbfmm_hip_pool_bytes() == 100 * MIB
    for p in ps:                                           # 1000 MiB more: 80 over the bound
        lib.wbfmm_hip_free(p)
    assert lib.wbfmm_hip_pool_bytes() == 900 * MIB         # the oldest that may go went
    lib.wbfmm_hip_debug_fail_mallocs(1)
    p = take(lib, MIB)                                     # tried again with what is released
    assert lib.wbfmm_hip_pool_bytes() == 100 * MIB
    assert hip.hipStreamEndCapture(s, ctypes.byref(g)) == 0
    assert hip.hipGraphGetNodes(g, None, ctypes.byref(nodes)) == 0 and nodes.value == 0
    assert hip.hipGraphDestroy(g) == 0
    lib.wbfmm_hip_free(p)
    assert lib.wbfmm_hip_stream_destroy(s) == 0
    assert lib.wbfmm_hip_pool_bytes() == MIB


def test_foreign_stream(wb, lib):
    """a stream of the caller's: nothing kept, and a block of the library's
    stream freed there goes back to the runtime"""
    hip = runtime()
    s = _vp()
    assert hip.hipStreamCreate(ctypes.byref(s)) == 0
    a = take(lib, MIB)
    wb.sync()
    lib.wbfmm_hip_set_stream(s, None)
    b = take(lib, MIB)
    lib.wbfmm_hip_free(b)
    lib.wbfmm_hip_free(a)
    assert lib.wbfmm_hip_pool_bytes() == 0
    lib.wbfmm_hip_set_stream(None, None)
    assert hip.hipStreamSynchronize(s) == 0 and hip.hipStreamDestroy(s) == 0


ADDRESS = r"""
import ctypes, sys
import wbfmm_amd as wb
L, MIB, foreign = wb.lib(), 1 << 20, sys.argv[1] == "1"
vp, sz = ctypes.c_void_p, ctypes.c_size_t
def take(n):
    p = vp()
    assert L.wbfmm_hip_malloc(ctypes.byref(p), n) == 0
    return p.value
wb.sync()
hip = ctypes.CDLL(next(l.split()[-1] for l in open("/proc/self/maps") if "libamdhip64" in l))
s, pool, back = vp(), vp(), 0
assert hip.hipStreamCreate(ctypes.byref(s)) == 0
assert hip.hipDeviceGetDefaultMemPool(ctypes.byref(pool), 0) == 0
for size in (2 * MIB, 16 * MIB, MIB // 4, 6 * MIB, 48 * MIB, MIB):
    a = take(size)
    wb.sync()
    assert hip.hipFree(vp(a)) == 0
    hip.hipMemPoolTrimTo(pool, sz(0))
    L.wbfmm_hip_set_stream(s if foreign else None, None)
    ps = [take(size // 2) for _ in range(8)]
    L.wbfmm_hip_set_stream(None, None)
    assert hip.hipStreamSynchronize(s) == 0
    if a in ps:
        back += 1
        L.wbfmm_hip_free(a)
        assert L.wbfmm_hip_pool_bytes() == (0 if foreign else size // 2), size
    for p in ps:
        if p != a:
            L.wbfmm_hip_free(p)
    wb.sync()
    L.wbfmm_hip_pool_release()
    wb.sync()
assert hip.hipStreamDestroy(s) == 0
print("back", back)
"""


@pytest.mark.parametrize("foreign", [False, True])
def test_address_that_comes_back_with_another_size(foreign):
    """a block that its holder gave to hipFree: a later, smaller one at the
    same address is kept with its own size, or, allocated on a caller's
    stream, not at all (in a process of its own, where the runtime's pool
    holds nothing else and gives the address back)"""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-u", "-c", ADDRESS, str(int(foreign))], cwd=root,
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
    if "back 0" in r.stdout:
        pytest.skip("the runtime gave the address to no later block")


def test_contents_in_stream_order(wb, lib):
    """a block handed out again while its last use is still queued"""
    n = 8 * MIB // 8
    want = np.arange(n, dtype=np.float64)
    for rep in range(8):
        a = wb.DeviceBuffer.from_array(want + rep)
        c = wb.DeviceBuffer(8 * n)
        assert lib.wbfmm_hip_memcpy(c.ptr, a.ptr, 8 * n) == 0   # device copy, queued
        was = a.ptr
        a.free()
        b = wb.DeviceBuffer(8 * n)
        assert b.ptr == was                                     # the same block
        b.zero()
        assert np.array_equal(c.download(np.zeros(n)), want + rep)
        assert not b.download(np.ones(n)).any()
        b.free()
        c.free()
        wb.sync()
        lib.wbfmm_hip_pool_release()    # the next freed block is the only one kept
