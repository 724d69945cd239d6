"""GPU: which plan a call takes, told by the device memory it allocates.

A handle with its own memory functions records every allocation.  A powm call's
scratch is R^2 mod m and the window table, whose size tells the lane layouts
and the matrix-core kernel apart."""
import ctypes
import json
import os

import numpy as np
import pytest

import xmp_amd
from helpers import O, assert_rows_equal, gmp, inputs
from xmp_amd import ext, hip

pytestmark = pytest.mark.gpu

_ALLOC = ctypes.CFUNCTYPE(ctypes.c_void_p, ctypes.c_size_t)
_FREE = ctypes.CFUNCTYPE(None, ctypes.c_void_p)


class Recording(xmp_amd.Handle):
    """A handle whose device allocations are listed in `sizes`."""

    def __init__(self):
        libc = ctypes.CDLL(None)
        libc.malloc.restype, libc.malloc.argtypes = ctypes.c_void_p, [ctypes.c_size_t]
        libc.free.argtypes = [ctypes.c_void_p]
        self.sizes = []

        def da(n):
            self.sizes.append(n)
            return hip.malloc(max(n, 1))

        self._fns = (_ALLOC(lambda n: libc.malloc(max(n, 1))), _FREE(libc.free), _ALLOC(da),
                     _FREE(lambda p: hip.free(p) if p else None))
        self.h = ctypes.c_void_p()
        rc = xmp_amd.lib().xmpHandleCreateWithMemoryFunctions(
            ctypes.byref(self.h), *[ctypes.cast(f, ctypes.c_void_p) for f in self._fns])
        assert rc == 0
        self._policy = None


@pytest.fixture
def recording():
    h = Recording()
    yield h
    h.close()


SHIPPED = os.path.join(os.path.dirname(xmp_amd.LIB_PATH), "tune_gfx950.json")


@pytest.fixture
def tables():
    yield lambda table: ext.tuner_load(json.dumps(table))
    with open(SHIPPED) as f:
        ext.tuner_load(f.read())


def _entry(bits, exp_bits, count, layout, window):
    lanes, digits, radix = layout
    return {"precision": bits, "exp_bits": exp_bits, "count": count, "lanes": lanes, "digits": digits, "radix": radix,
            "window": window, "ms": 1.0, "powm_per_s": 1.0}


def _r2_bytes(bits, n):
    return 4 * (bits // 32) * (-(-n // 64) * 64)


def _lane_bytes(layout, n, window):
    return 4 * ((-(-n // 64) * 64) << window) * layout[0] * layout[1]


def _mx_bytes(bits, n, window):
    return 4 * (n << window) * 4 * (bits // 128)   # (sizes of a whole number of compiled blocks)


def _powm(h, bits, exp_bits, n):
    """One call, checked; the device memory that it allocated."""
    m, b, e = inputs.powm_class(8100 + bits, n, bits, exp_bits=exp_bits)
    M, B, E, out = h.from_array(m), h.from_array(b), h.from_array(e), h.integers(bits, n)
    h.sizes.clear()
    h.powm(out, B, E, M)
    sizes = list(h.sizes)
    assert_rows_equal(out.get(), gmp(O.GO_POWM, n, bits // 32, b, e, m), "%d x %d bits" % (n, bits))
    for x in (M, B, E, out):
        x.close()
    return sizes


@pytest.mark.parametrize("bits,layout", [(1024, (16, 3, 28)), (3072, (4, 28, 28)), (4096, (4, 37, 28))])
def test_a_loaded_table_decides(recording, tables, bits, layout):
    """A program's own table decides the plain call of a precision that it
    lists; others, and the shipped table's, go to the matrix cores first."""
    n, exp_bits, window = 100, 96, 3
    tables({"device": "gfx950", "entries": [_entry(bits, exp_bits, n, layout, window)]})
    assert _powm(recording, bits, exp_bits, n) == [_r2_bytes(bits, n) + _lane_bytes(layout, n, window)]
    assert _powm(recording, 2048, exp_bits, 3 * n) == [_r2_bytes(2048, 3 * n) + _mx_bytes(2048, 3 * n, window)]
    with open(SHIPPED) as f:
        ext.tuner_load(f.read())
    n = 700   # (the scratch of the calls before is too short)
    assert _powm(recording, bits, exp_bits, n) == [_r2_bytes(bits, n) + _mx_bytes(bits, n, window)]


def test_a_loaded_table_decides_for_batches(recording, tables):
    """The classes of a mixed batch that a program's table lists run in the
    persistent queue, the others on the matrix cores."""
    sizes, counts, exp_bits, window = (1024, 4096), (70, 30), 96, 3
    tables({"device": "gfx950", "entries": [_entry(4096, exp_bits, 30, (4, 38, 27), window)]})
    arrays, wants = [], []
    for bits, c in zip(sizes, counts):
        m, b, e = inputs.powm_class(8300 + bits, c, bits, exp_bits=exp_bits)
        wants.append(gmp(O.GO_POWM, c, bits // 32, b, e, m))
        arrays.append([recording.integers(bits, c)] + [recording.from_array(x) for x in (b, e, m)])
    recording.sizes.clear()
    batch = ext.Batch(recording, *[[a[k] for a in arrays] for k in range(4)], list(counts))
    assert _mx_bytes(1024, 70, window) in recording.sizes
    assert _lane_bytes((4, 38, 27), 30, window) in recording.sizes
    assert _mx_bytes(4096, 30, window) not in recording.sizes
    for _ in range(2):
        batch.launch_async()
        for a, want, bits in zip(arrays, wants, sizes):
            assert_rows_equal(a[0].get(), want, "batched %d-bit class" % bits)
    batch.close()
    for a in arrays:
        for x in a:
            x.close()


def test_a_long_chain_beside_many_short_ones(recording):
    """A class of which one tile takes longer than the queue's whole load goes to
    the matrix cores however many instances the other classes have; with as
    many long ones it does not."""
    for shapes, matrix in ((((1536, 32, 8000), (1024, 1024, 200)), True), (((1024, 1024, 60000), (1024, 1024, 200)), False)):
        arrays, wants = [], []
        for bits, exp_bits, c in shapes:
            m, b, e = inputs.powm_class(8350 + bits + c, c, bits, exp_bits=exp_bits)
            if c > 200:
                m, b, e = (np.tile(x[:100], (c // 100, 1)) for x in (m, b, e))
            wants.append(gmp(O.GO_POWM, 100, bits // 32, b[:100], e[:100], m[:100]))
            arrays.append([recording.integers(bits, c)] + [recording.from_array(x) for x in (b, e, m)])
        recording.sizes.clear()
        batch = ext.Batch(recording, *[[a[k] for a in arrays] for k in range(4)], [c for _, _, c in shapes])
        assert any(_mx_bytes(1024, 200, w) in recording.sizes for w in range(2, 8)) == matrix
        for _ in range(2):
            batch.launch_async()
            for a, want in zip(arrays, wants):
                got = a[0].get()
                assert_rows_equal(got[:100], want, "first instances")
                if got.shape[0] > 200:
                    assert_rows_equal(got[-100:], want, "last instances")
        batch.close()
        for a in arrays:
            for x in a:
                x.close()


@pytest.mark.parametrize("bits,n", [(1024, 300), (3072, 50)])
def test_digitmp_takes_the_default_plan(recording, bits, n):
    """The digit-serial policy is accepted and treated as the default one."""
    plans = []
    for alg, k in ((xmp_amd.ALG_DEFAULT, n), (xmp_amd.ALG_DIGITMP, 2 * n)):   # (scratch only grows)
        recording.set_algorithm(alg)
        plans.append(_powm(recording, bits, 96, k))
        assert plans[-1] == [_r2_bytes(bits, k) + _mx_bytes(bits, k, 3)]


@pytest.mark.parametrize("bits", [5120, 6144, 8192])
def test_long_moduli_take_no_division_workspace(recording, bits):
    """R^2 mod m of the matrix-core kernel is a division in LDS."""
    assert _powm(recording, bits, 96, 40) == [_r2_bytes(bits, 40) + _mx_bytes(bits, 40, 3)]


@pytest.mark.parametrize("la,lb,uses", [
    (300, 150, False),     # signed digits
    (2080, 1040, False),
    (2200, 1100, False),   # a wave's LDS: longer divisors, and dividends too long for the rows
    (9000, 300, False),
    (8001, 8000, True),    # neither holds it
])
def test_division_allocates_what_its_kernel_uses(recording, la, lb, uses):
    """A limit still refuses by the sizes alone."""
    h, n = recording, 40
    a, b = inputs.uniform(8500 + la, n, la), inputs.uniform(8501 + lb, n, lb)
    b[:, -1] |= np.uint32(0x80000000)
    A, B, Q, R = h.from_array(a), h.from_array(b), h.integers(32 * la, n), h.integers(32 * lb, n)
    words = (2 * lb + 1) * 256
    h.sizes.clear()
    h.divmod(Q, R, A, B)
    assert h.sizes == ([4 * words] if uses else [])
    wq, wr = gmp(O.GO_DIV, n, la, a, b, out2_limbs=lb)
    assert_rows_equal(Q.get(), wq, "q")
    assert_rows_equal(R.get(), wr, "r")
    h.set_scratch_limit(4 * words - 1)
    with pytest.raises(xmp_amd.XmpError) as err:
        h.divmod(Q, R, A, B)
    assert err.value.code == xmp_amd.INCREASE_SCRATCH_LIMIT
    h.set_scratch_limit(0)
    for x in (A, B, Q, R):
        x.close()


def test_short_transfers_take_no_scratch(recording):
    """Imports and exports through the handle's pinned slots; a limit below
    their size still refuses them."""
    h, n, limbs = recording, 50, 20
    a = inputs.uniform(8600, n, limbs)
    x = h.integers(32 * limbs, n)
    h.sizes.clear()
    x.load(a)
    assert np.array_equal(x.get(), a)
    assert h.sizes == []
    h.set_scratch_limit(4 * n * limbs - 1)
    for call in (lambda: x.load(a), x.get):
        with pytest.raises(xmp_amd.XmpError) as err:
            call()
        assert err.value.code == xmp_amd.INCREASE_SCRATCH_LIMIT
    h.set_scratch_limit(0)
    x.close()


@pytest.mark.parametrize("n,scratch_in,scratch_out", [(100, False, False), (103, False, True), (513, True, True)])
@pytest.mark.parametrize("fmt", [(-1, 2, 1), (1, 2, -1), (-1, 8, 1), (1, 8, -1)])   # (order, size, endian)
def test_formats_of_no_whole_words(recording, fmt, n, scratch_in, scratch_out):
    """Formats that the kernels handle a short word or a byte at a time are
    transposed in device scratch, not across the bus, above 40 KiB in and 8 KiB
    out (24 as 64-bit words)."""
    scratch_out = scratch_out and (fmt[1] != 8 or n > 300)
    h, limbs, (order, size, endian) = recording, 20, fmt
    a = inputs.uniform(8700, n, limbs)
    words = a.astype("<u4").view("<u%d" % size).reshape(n, -1)
    host = np.ascontiguousarray(words[:, ::-order].astype((">" if endian == 1 else "<") + "u%d" % size))
    L, x = xmp_amd.lib(), h.integers(32 * limbs, n)
    h.sizes.clear()
    assert L.xmpIntegersImport(h.h, x.x, words.shape[1], order, size, endian, 0, host.ctypes.data, n) == 0
    assert h.sizes == ([4 * n * limbs] if scratch_in else [])
    assert np.array_equal(x.get(), a)
    back, got = np.zeros_like(host), ctypes.c_uint32()
    assert L.xmpIntegersExport(h.h, back.ctypes.data, ctypes.byref(got), order, size, endian, 0, x.x, n) == 0
    assert h.sizes == ([4 * n * limbs] if scratch_in or scratch_out else [])
    assert got.value == words.shape[1] and back.tobytes() == host.tobytes()
    x.close()


@pytest.mark.parametrize("limbs,n,uses", [(1, 65536, False), (2, 28672, False), (2, 28700, True), (8, 1792, False),
                                          (8, 1800, True), (11, 950, True), (12, 850, False), (16, 700, True)])
def test_imports_of_short_integers_of_no_whole_words(recording, limbs, n, uses):
    """The slot keeps 448 KiB by the limbs, 40 from 12 limbs on, and more than
    that is transposed in scratch."""
    a = inputs.uniform(8750 + limbs, n, limbs)
    host = np.ascontiguousarray(a.astype("<u4").view("<u2").astype(">u2"))   # 16-bit big-endian words, low one first
    x = recording.integers(32 * limbs, n)
    recording.sizes.clear()
    assert xmp_amd.lib().xmpIntegersImport(recording.h, x.x, 2 * limbs, -1, 2, 1, 0, host.ctypes.data, n) == 0
    assert recording.sizes == ([4 * n * limbs] if uses else [])
    assert np.array_equal(x.get(), a)
    x.close()


@pytest.mark.parametrize("limbs,n,uses", [(9, 56, False), (9, 60, True), (33, 124, True), (33, 125, False), (7, 300, False),
                                          (36, 100, False), (65, 32, False), (65, 33, True)])
def test_short_imports_of_odd_lengths(recording, limbs, n, uses):
    """Tiles of 2 to 16 KiB, but for a few rows, are read from device scratch,
    not across the bus."""
    a = inputs.uniform(8800 + limbs, n, limbs)
    x = recording.integers(32 * limbs, n)
    recording.sizes.clear()
    x.load(a)
    assert recording.sizes == ([4 * n * limbs] if uses else [])
    assert np.array_equal(x.get(), a)
    x.close()


def test_more_products_than_a_grid_of_waves_holds(fresh_handle):
    """2^26 and some squares of 129 limbs, truncated and of repeated operands: a
    wave each would be 2^32 threads."""
    h, limbs, n = fresh_handle, 129, (1 << 26) + 100
    a = inputs.uniform(8900, 3, limbs)
    want = gmp(O.GO_MUL, 3, limbs, a, a)
    A, P = h.from_array(a), h.integers(32 * limbs, n)
    h.mul(P, A, A, n)
    rows = np.array([0, 1, 2, 63, 64, 65535, n // 2, n - 65, n - 64, n - 2, n - 1], np.uint32)
    out = h.integers(32 * limbs, rows.size)
    h.set_indices(1, rows)
    try:
        assert xmp_amd.lib().xmpIntegersSet(h.h, out.x, P.x, rows.size) == 0
    finally:
        h.clear_indices()
    assert_rows_equal(out.get(), want[rows % 3], "repeated squares")
    for x in (A, P, out):
        x.close()


def _sample(h, x, rows):
    """Some instances of a batch too long to export."""
    out = h.integers(x.precision, rows.size)
    h.set_indices(1, rows)
    try:
        assert xmp_amd.lib().xmpIntegersSet(h.h, out.x, x.x, rows.size) == 0
    finally:
        h.clear_indices()
    got = out.get()
    out.close()
    return got


def test_more_long_products_than_a_grid_of_workgroups_holds(fresh_handle):
    """2^25 and some products of 513 limbs by one, truncated and of repeated
    operands: two waves each would be 2^32 threads."""
    h, limbs, n = fresh_handle, 513, (1 << 25) + 100
    a, b = inputs.uniform(8950, 3, limbs), inputs.uniform(8951, 1, 1)
    A, B, P = h.from_array(a), h.from_array(b), h.integers(32 * limbs, n)
    h.mul(P, A, B, n)
    rows = np.array([0, 1, 2, 63, 64, 65535, n // 2, n - 101, n - 65, n - 64, n - 2, n - 1], np.uint32)
    assert_rows_equal(_sample(h, P, rows), gmp(O.GO_MUL, 3, limbs, a, np.repeat(b, 3, axis=0))[rows % 3], "products")
    for x in (A, B, P):
        x.close()


def test_more_divisions_than_a_grid_of_lane_groups_holds(fresh_handle):
    """2^30 and some divisions by 67 limbs, of repeated operands: four lanes
    each would be 2^32 threads."""
    h, n = fresh_handle, (1 << 30) + 100
    a, b = inputs.uniform(8960, 5, 1), np.zeros((1, 67), np.uint32)
    b[0, 0] = 12345
    A, B, Q = h.from_array(a), h.from_array(b), h.integers(32, n)
    h.div(Q, A, B, n)
    rows = np.array([0, 1, 2, 63, 64, 65535, n // 2, n - 101, n - 65, n - 64, n - 2, n - 1], np.uint32)
    assert np.array_equal(_sample(h, Q, rows)[:, 0], (a[:, 0] // 12345)[rows % 5])
    for x in (A, B, Q):
        x.close()


@pytest.mark.parametrize("bits", [1024, 2048, 6144])
def test_a_limit_below_the_lanes_plan_refuses(recording, bits):
    """One instance's table is short on the matrix cores; the limits that are
    refused are those of a lane layout's, of 64 instances."""
    h = recording
    h.set_scratch_limit(_r2_bytes(bits, 1) + _mx_bytes(bits, 1, 3))
    with pytest.raises(xmp_amd.XmpError) as err:
        _powm(h, bits, 96, 1)
    assert err.value.code == xmp_amd.INCREASE_SCRATCH_LIMIT
    h.set_scratch_limit(0)
    assert _powm(h, bits, 96, 1) == [_r2_bytes(bits, 1) + _mx_bytes(bits, 1, 3)]
