"""Device memory behind tsp_malloc / tsp_free: freed blocks are handed out
again only when nothing uses them, whole, and can be given back."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip(tsp):
    if not tsp.device_available():
        pytest.fail("no gfx950 device: GPU tests need an MI355X")
    return tsp.load()[0]


def alloc(hip, n):
    p = C.c_void_p()
    assert hip.tsp_malloc(C.byref(p), n) == 0
    return p.value


@pytest.mark.parametrize("size", [1, 4096, 4097, 1 << 20, (1 << 20) + 1, 100 << 20])
def test_block_comes_back(hip, size):
    assert hip.tsp_mem_trim() == 0
    a, b = alloc(hip, size), alloc(hip, size)
    assert a != b
    assert hip.tsp_free(a) == 0
    assert alloc(hip, size) == a                    # the one idle block of its size
    big = alloc(hip, 4 * size + (1 << 20))
    assert hip.tsp_free(a) == 0 and hip.tsp_free(b) == 0 and hip.tsp_free(big) == 0
    assert alloc(hip, max(size // 2, 1)) != big     # too large for it
    host = np.full(size, 7, np.uint8)
    c = alloc(hip, size)
    assert hip.tsp_memcpy_h2d(c, host.ctypes.data_as(C.c_void_p), size) == 0
    back = np.zeros(size, np.uint8)
    assert hip.tsp_memcpy_d2h(back.ctypes.data_as(C.c_void_p), c, size) == 0
    assert np.array_equal(back, host)
    assert hip.tsp_free(c) == 0 and hip.tsp_mem_trim() == 0
    assert hip.tsp_free(None) == 0


def test_free_waits_for_other_streams(hip):
    n = 512 << 20
    s = C.c_void_p()
    assert hip.tsp_stream_create_nonblocking(C.byref(s)) == 0
    src, dst = alloc(hip, n), alloc(hip, n)
    assert hip.tsp_memset(src, 5, n) == 0
    for _ in range(8):
        assert hip.tsp_copy_kernel(dst, src, n, s) == 0
    assert hip.tsp_free(src) == 0                   # still being read
    again = alloc(hip, n)
    assert again == src
    assert hip.tsp_memset(again, 9, n) == 0
    back = np.zeros(n, np.uint8)
    assert hip.tsp_memcpy_d2h(back.ctypes.data_as(C.c_void_p), dst, n) == 0
    assert int(back.min()) == 5 and int(back.max()) == 5
    for p in (again, dst):
        assert hip.tsp_free(p) == 0
    assert hip.tsp_stream_destroy(s) == 0 and hip.tsp_mem_trim() == 0


def test_threads_never_share_a_block(hip):
    errors = []

    def work(k):
        rng = np.random.default_rng(k)
        for i in range(40):
            n = int(rng.integers(1, 1 << 18))
            p = alloc(hip, n)
            want = np.full(n, (k * 40 + i) % 251, np.uint8)
            got = np.zeros(n, np.uint8)
            hip.tsp_memcpy_h2d(p, want.ctypes.data_as(C.c_void_p), n)
            hip.tsp_memcpy_d2h(got.ctypes.data_as(C.c_void_p), p, n)
            if not np.array_equal(got, want):
                errors.append((k, i))
            if hip.tsp_free(p) != 0:
                errors.append((k, i, "free"))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    assert hip.tsp_mem_trim() == 0
