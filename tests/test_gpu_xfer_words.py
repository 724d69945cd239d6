"""GPU: imports and exports of whole-word formats (least or most significant
first, little- or big-endian, words of any size), which move as blocks of
4 x 4 words, as LDS tiles (limb counts that are not a multiple of four,
buffers off 16-byte alignment) or word by word, against numpy.  Batches that
end inside a block leave the instances past them as they were."""
import ctypes

import numpy as np
import pytest

import xmp_amd
from helpers import inputs

pytestmark = pytest.mark.gpu

# (word size, order, endian); the last two mix orders and stay word by word
FORMATS = [(4, -1, -1), (4, 1, -1), (4, -1, 1), (4, 1, 1), (1, -1, 1), (1, 1, -1), (2, -1, -1), (2, 1, 1), (8, -1, -1),
           (8, 1, 1), (8, 1, -1), (2, -1, 1)]


def _compact(x, size, order, endian):
    """x (count, limbs, little-endian limbs) as words of `size` bytes."""
    w = np.ascontiguousarray(x).view(np.uint8).reshape(x.shape[0], -1, size)
    if endian == 1:
        w = w[:, :, ::-1]
    if order == 1:
        w = w[:, ::-1]
    return np.ascontiguousarray(w).reshape(x.shape[0], -1)


@pytest.mark.parametrize("limbs", [1, 3, 4, 8, 9, 10, 12, 20, 33, 64, 68, 132])
@pytest.mark.parametrize("count", [1, 3, 66, 257])
def test_word_formats(handle, limbs, count):
    L = xmp_amd.lib()
    x = inputs.uniform(8000 + limbs + count, count + 3, limbs)
    old = inputs.uniform(8001 + limbs + count, count + 3, limbs)
    X = handle.from_array(old)
    for size, order, endian in FORMATS:
        if 4 * limbs % size:
            continue
        words = 4 * limbs // size
        src = _compact(x, size, order, endian)
        X.load(old)
        for at in (0, 4):   # 16-byte aligned or not (host buffers are staged aligned; device ones are used as they are)
            room = src.nbytes + 64
            dev = xmp_amd_hip_malloc(room)
            try:
                base = (dev + 15) // 16 * 16 + at
                _hip().memcpy_htod(base, src)
                xmp_amd.check(L.xmpIntegersImport(handle.h, X.x, words, order, size, endian, 0, base, count), "import")
                got = X.get()
                assert np.array_equal(got[:count], x[:count]), (size, order, endian, at)
                assert np.array_equal(got[count:], old[count:]), (size, order, endian, at)
                _hip().memcpy_htod(base, np.zeros_like(src))
                xmp_amd.check(L.xmpIntegersExport(handle.h, base, None, order, size, endian, 0, X.x, count), "export")
                back = np.empty((count, 4 * limbs), np.uint8)
                _hip().hip().hipMemcpy(ctypes.c_void_p(back.ctypes.data), ctypes.c_void_p(base), back.nbytes, 2)
                assert np.array_equal(back, src[:count]), (size, order, endian, at)
            finally:
                _hip().free(dev)
        host = np.zeros((count, 4 * limbs), np.uint8)
        xmp_amd.check(L.xmpIntegersExport(handle.h, host.ctypes.data, None, order, size, endian, 0, X.x, count), "export")
        assert np.array_equal(host, src[:count]), (size, order, endian, "host")
    X.close()


def _hip():
    from xmp_amd import hip
    return hip


def xmp_amd_hip_malloc(nbytes):
    return _hip().malloc(nbytes, 0)
