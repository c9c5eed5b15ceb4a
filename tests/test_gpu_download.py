"""iris_hip_download: copies into pinned memory on the side stream, each behind
what the library stream was given before it and waited for by its slot."""
import ctypes

import numpy as np
import pytest

import iris_testlib as tl

pytestmark = pytest.mark.gpu
N = 1 << 20


@pytest.fixture(scope="module")
def lib():
    lib = tl.hip()
    lib.iris_hip_host_malloc.restype = ctypes.c_void_p
    lib.iris_hip_host_malloc.argtypes = [ctypes.c_size_t]
    lib.iris_hip_host_free.argtypes = [ctypes.c_void_p]
    lib.iris_hip_download.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
    lib.iris_hip_download_wait.argtypes = [ctypes.c_int]
    lib.iris_hip_memcpy_d2d.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t]
    return lib


def test_order_and_slots(lib):
    """Every slot twice: a download sees all work enqueued before it (a chain
    of device copies that ends in its source) and none of the later work on
    other memory waits for or disturbs it; a slot's second download replaces
    the first."""
    host = lib.iris_hip_host_malloc(8 * N * 4)
    assert host, lib.iris_hip_last_error()
    view = np.ctypeslib.as_array((ctypes.c_uint32 * (8 * N)).from_address(host)).reshape(8, N)
    rng = np.random.default_rng(5)
    data = rng.integers(0, 1 << 32, (3, N), dtype=np.uint32)
    src, tmp = [tl.Dev.of(d) for d in data], tl.Dev(N * 4)
    out = [tl.Dev(N * 4) for _ in range(8)]
    for turn in range(2):
        view[:] = 0
        for s in range(8):
            for k in range(21):     # the last of them is what the download must see
                assert lib.iris_hip_memcpy_d2d(tmp.ptr, src[(k + s + turn) % 3].ptr, N * 4) == 0
            assert lib.iris_hip_memcpy_d2d(out[s].ptr, tmp.ptr, N * 4) == 0
            assert lib.iris_hip_download(host + s * N * 4, out[s].ptr, N * 4, s) == 0, lib.iris_hip_last_error()
        for s in reversed(range(8)):
            assert lib.iris_hip_download_wait(s) == 0
            assert np.array_equal(view[s], data[(20 + s + turn) % 3]), (turn, s)
    assert lib.iris_hip_download_wait(3) == 0     # done already
    assert lib.iris_hip_sync() == 0
    lib.iris_hip_host_free(host)


def test_bad_arguments(lib):
    """Slots outside 0..7 and missing memory are refused before anything is enqueued."""
    d, host = tl.Dev(4096), lib.iris_hip_host_malloc(4096)
    for slot in (-1, 8, 1000):
        assert lib.iris_hip_download(host, d.ptr, 4096, slot) == -1
        assert lib.iris_hip_download_wait(slot) == -1
    assert lib.iris_hip_download(None, d.ptr, 4096, 0) == -1
    assert lib.iris_hip_download(host, None, 4096, 0) == -1
    lib.iris_hip_host_free(host)
