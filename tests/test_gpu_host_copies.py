"""GPU: synchronous transfers between host memory and the GPU, which pass
through a handle's pinned slots in chunks: sizes at the edges of the chunks and
of the ring of slots, pinned and pageable memory, a handle whose stream
changes between calls, and two handles on two threads."""
import threading

import numpy as np
import pytest
import torch

import xmp_amd
from helpers import inputs

pytestmark = pytest.mark.gpu

KIB = 1024
# one chunk, both sides of a half slot, of 1 MiB (whole slots from there), of the ring, and a ragged end
SIZES = [4, 256 * KIB, 256 * KIB + 4, KIB * KIB, KIB * KIB + 4, 2 * KIB * KIB, 2 * KIB * KIB + 512 * KIB + 4, 5 * KIB * KIB - 4]


def _round_trip(h, x, dst=None):
    L, n = xmp_amd.lib(), x.shape[0]
    X = h.integers(32 * x.shape[1], n)
    xmp_amd.check(L.xmpIntegersImport(h.h, X.x, x.shape[1], -1, 4, -1, 0, x.ctypes.data, n), "import")
    out = np.zeros_like(x) if dst is None else dst
    xmp_amd.check(L.xmpIntegersExport(h.h, out.ctypes.data, None, -1, 4, -1, 0, X.x, n), "export")
    X.close()
    return out


@pytest.mark.parametrize("nbytes", SIZES)
@pytest.mark.parametrize("pinned", [False, True])
def test_sizes(handle, nbytes, pinned):
    x = inputs.uniform(8300 + nbytes % 97, nbytes // 4, 1)
    if pinned:
        a, b = (torch.empty(x.shape, dtype=torch.int32, pin_memory=True).numpy().view(np.uint32) for _ in range(2))
        a[:] = x
        assert np.array_equal(_round_trip(handle, a, b), x)
    else:
        assert np.array_equal(_round_trip(handle, x), x)


def test_streams_in_turn(fresh_handle):
    s, t = torch.cuda.Stream(), torch.cuda.Stream()
    for k in range(6):
        fresh_handle.set_stream((s, t)[k % 2].cuda_stream)
        x = inputs.uniform(8400 + k, 300000 + 4096 * k, 1)
        assert np.array_equal(_round_trip(fresh_handle, x), x)


def test_indexed_export_keeps_unselected_rows(fresh_handle):
    h, n = fresh_handle, 40000
    x = inputs.uniform(8500, n, 8)
    X = h.from_array(x)
    idx = np.arange(0, 2 * n, 2, dtype=np.uint32)
    h.set_indices(0, idx)
    out = np.full((2 * n, 8), 0xA5A5A5A5, np.uint32)
    xmp_amd.check(xmp_amd.lib().xmpIntegersExport(h.h, out.ctypes.data, None, -1, 4, -1, 0, X.x, n), "export")
    h.clear_indices()
    assert np.array_equal(out[::2], x)
    assert (out[1:-1:2] == 0xA5A5A5A5).all()
    X.close()


def test_compare_and_popcount_results(handle):
    n = 300000
    a, b = inputs.uniform(8600, n, 1), inputs.uniform(8601, n, 1)
    A, B = handle.from_array(a), handle.from_array(b)
    assert np.array_equal(np.sign(handle.cmp(A, B)), np.sign(a[:, 0].astype(np.int64) - b[:, 0].astype(np.int64)))
    bits = np.unpackbits(a.view(np.uint8), axis=1).sum(axis=1)
    assert np.array_equal(handle.popc(A), bits)
    A.close()
    B.close()


def test_two_handles_on_two_threads():
    bad = []

    def work(seed):
        with xmp_amd.Handle() as h:
            s = torch.cuda.Stream()
            h.set_stream(s.cuda_stream)
            for k in range(8):
                x = inputs.uniform(seed + k, 100000 * (1 + k % 4), 2)
                if not np.array_equal(_round_trip(h, x), x):
                    bad.append((seed, k))

    threads = [threading.Thread(target=work, args=(8700 + 50 * i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
