"""GPU: a buffer copied out to pinned memory by a kernel (tlhip_copy_to_host): every byte and none past the last, for whole
and broken 16 bytes and more than one pass of the grid; replayed in a graph; other targets refused on the host."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture
def pinned(lib):
    p = C.c_void_p()
    assert lib.c.tlhip_host_alloc(C.byref(p), (4 << 20) + 64) == 0
    yield np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_uint8)), shape=((4 << 20) + 64,))
    lib.c.tlhip_host_free(p)


@pytest.mark.parametrize("nbytes", [1, 15, 16, 17, 4095, 4096, 4100, 607744, (4 << 20) - 1, (4 << 20) + 33])
def test_bytes(lib, pinned, nbytes):
    data = np.random.default_rng(nbytes).integers(0, 256, nbytes, dtype=np.uint8)
    dev = lib.to_device(data)
    pinned[:] = 0xA5
    assert lib.c.tlhip_copy_to_host(pinned.ctypes.data, dev.ptr, nbytes) == 0
    lib.sync()
    assert np.array_equal(pinned[:nbytes], data) and np.all(pinned[nbytes:] == 0xA5)
    dev.free()


def test_replays(lib, pinned):
    dev = lib.to_device(np.zeros(1000, np.float32))
    lib.graph_begin()
    rc = lib.c.tlhip_copy_to_host(pinned.ctypes.data, dev.ptr, 4000)
    g = lib.graph_end()
    assert rc == 0
    for i in range(4):
        lib.c.tlhip_fill_u32(dev.ptr, i + 1, 1000)
        lib.graph_launch(g)
        lib.sync()
        assert np.all(pinned[:4000].view(np.uint32) == i + 1)
    lib.graph_destroy(g)
    dev.free()


def test_refused(lib, pinned):
    dev, other = lib.to_device(np.zeros(64, np.float32)), lib.to_device(np.zeros(64, np.float32))
    pageable = np.zeros(128, np.float32)
    at = pageable.ctypes.data + (-pageable.ctypes.data) % 16
    for dst, src in ((at, dev.ptr), (other.ptr, dev.ptr), (pinned.ctypes.data + 4, dev.ptr), (None, dev.ptr), (pinned.ctypes.data, None)):
        assert lib.c.tlhip_copy_to_host(dst, src, 64) != 0
    assert lib.c.tlhip_copy_to_host(pinned.ctypes.data, dev.ptr, 0) == 0
    dev.free(); other.free()
