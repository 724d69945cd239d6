"""GPU: the Montgomery lane layouts themselves, whichever kernel the plain call
takes, against GMP.

A Montgomery context always runs the layout that it reports."""
import json
import os

import numpy as np
import pytest

import xmp_amd
from helpers import O, assert_rows_equal, gmp, inputs
from xmp_amd import ext

pytestmark = pytest.mark.gpu

EXP_BITS = 96


def _load(layout, bits, count):
    lanes, digits, radix = layout
    entry = {"precision": bits, "exp_bits": EXP_BITS, "count": count, "lanes": lanes, "digits": digits,
             "radix": radix, "window": 3, "ms": 1.0, "powm_per_s": 1.0}
    assert xmp_amd.lib().xmpTunerLoad(json.dumps({"device": "gfx950", "entries": [entry]}).encode()) == 0


@pytest.fixture
def tables():
    """Lets a test load layout tables; the shipped one is back afterwards."""
    yield _load
    with open(os.path.join(os.path.dirname(xmp_amd.LIB_PATH), "tune_gfx950.json")) as f:
        assert xmp_amd.lib().xmpTunerLoad(f.read().encode()) == 0


def _edge_case(seed, n, bits):
    m, b, e = inputs.powm_class(seed, n, bits, exp_bits=EXP_BITS)
    ones = np.uint32(0xFFFFFFFF)
    m[0], b[0], b[0, 0], e[0] = ones, ones, ones - 1, ones   # 2^bits - 1, base m - 1
    m[1] = 0
    m[1, 0] = 1                                              # m = 1
    m[2] = 0
    m[2, 0], b[2] = 3, ones                                  # a base far above the modulus
    m[3] = 0
    m[3, 0], m[3, -1], b[3] = 1, 0x80000000, ones            # 2^(bits-1) + 1
    m[4, -1], b[4] = 0, ones                                 # a leading zero limb, the largest base
    m[5, m.shape[1] // 2:], b[5] = 0, ones                   # the upper half zero
    e[6] = 0
    b[7] = 0
    m[8, 0] &= ones - 1                                      # even
    m[9] = 0
    want = np.zeros_like(m)
    odd = (m[:, 0] & 1).astype(bool)
    want[odd] = gmp(O.GO_POWM, int(odd.sum()), bits // 32, b[odd], e[odd], m[odd])
    return m, b, e, want


def _context_powm(handle, layout, bits, m, b, e, want):
    n = m.shape[0]
    M, B, E, out = handle.from_array(m), handle.from_array(b), handle.from_array(e), handle.integers(bits, n)
    ctx = ext.Montgomery(handle, M, EXP_BITS, n)
    try:
        assert tuple(ctx.layout()[:3]) == layout
        ctx.powm_async(out, B, E, n)
        assert_rows_equal(out.get(), want, "%dx%d radix %d, %d bits" % (layout + (bits,)))
    finally:
        ctx.close()
        for x in (M, B, E, out):
            x.close()


# (lanes, digits, radix): sizes at the layout's end and inside it, and sizes
# that leave the top lane nearly empty
LAYOUTS = {
    (1, 5, 28): (128, 96), (1, 10, 28): (256,), (1, 12, 28): (320,), (1, 20, 28): (512, 544), (1, 28, 28): (768,),
    (1, 37, 28): (1024,), (2, 19, 28): (1056, 1024, 544), (2, 28, 28): (1536, 1056), (2, 37, 28): (2048, 1088),
    (4, 19, 28): (2080, 1056), (4, 28, 28): (3072, 3104), (2, 55, 28): (3072,), (4, 37, 28): (4096, 3968, 3072),
    (4, 38, 27): (4096, 3968), (8, 19, 27): (4096, 3968, 2080), (8, 29, 27): (6144,), (8, 37, 28): (8192, 4160),
    (8, 38, 27): (8192, 4096), (16, 19, 27): (8192, 4096), (4, 10, 28): (1088, 1056), (8, 5, 28): (1088, 1056),
    (8, 10, 28): (2208, 1056), (16, 5, 28): (2208, 1056), (16, 3, 28): (1312, 1056), (32, 20, 26): (12288, 4096),
    (64, 20, 26): (20480,),
}
UNBATCHED = {(2, 55, 28), (4, 10, 28), (8, 5, 28), (8, 10, 28), (16, 5, 28), (16, 3, 28), (8, 37, 28)}


@pytest.mark.parametrize("layout", sorted(LAYOUTS))
def test_edges_of_every_layout(handle, tables, layout):
    """All ones, m = 1, small and even moduli, leading zero limbs, bases above
    the modulus, e = 0: in a plain call, in place, in a context and, where the
    persistent queue runs the layout, beside another class of a batch."""
    n = max(2 * (64 // layout[0]) + 1, 12)
    for bits in LAYOUTS[layout]:
        m, b, e, want = _edge_case(bits + layout[0], n, bits)
        tables(layout, bits, n)
        what = "%dx%d radix %d, %d bits" % (layout + (bits,))
        _context_powm(handle, layout, bits, m, b, e, want)
        M, B, E, out = handle.from_array(m), handle.from_array(b), handle.from_array(e), handle.integers(bits, n)
        handle.powm(out, B, E, M)
        assert_rows_equal(out.get(), want, what)
        if layout not in UNBATCHED:
            out.load(np.zeros_like(m))
            other = [handle.integers(16384, 1)] + [handle.from_array(x) for x in inputs.powm_class(5, 1, 16384, exp_bits=32)]
            batch = ext.Batch(handle, [out, other[0]], [B, other[2]], [E, other[3]], [M, other[1]], [n, 1])
            try:
                for _ in range(2):
                    batch.launch_async()
                    assert_rows_equal(out.get(), want, what + ", batched")
            finally:
                batch.close()
            for x in other:
                x.close()
        handle.powm(B, B, E, M)
        assert_rows_equal(B.get(), want, what + ", in place")
        for x in (M, B, E, out):
            x.close()


@pytest.mark.parametrize("layout,bits", [((1, 37, 28), 1024), ((2, 37, 28), 2048), ((4, 37, 28), 4096), ((8, 37, 28), 8192)])
def test_shared_and_gathered_operands_on_the_lanes(handle, tables, layout, bits):
    n, k = 2 * (64 // layout[0]) + 3, 5
    m, b, e, _ = _edge_case(bits, 14, bits)
    m[8:10] = inputs.odd_moduli(bits, 2, bits // 32)   # (none even)
    tables(layout, bits, n)
    rng = np.random.default_rng(bits)
    im, ib, io = rng.integers(0, 14, n).astype(np.uint32), rng.integers(0, 14, n).astype(np.uint32), rng.permutation(n).astype(np.uint32)
    M, B, E, out = handle.from_array(m), handle.from_array(b), handle.from_array(e[:k]), handle.integers(bits, n)
    rows = np.arange(n)
    handle.powm(out, B, E, M, n)
    assert_rows_equal(out.get(), gmp(O.GO_POWM, n, bits // 32, b[rows % 14], e[rows % k], m[rows % 14]), "shared")
    for which, idx in ((0, io), (1, ib), (3, im)):
        handle.set_indices(which, idx)
    try:
        handle.powm(out, B, E, M, n)
    finally:
        handle.clear_indices()
    assert_rows_equal(out.get()[io], gmp(O.GO_POWM, n, bits // 32, b[ib], e[rows % k], m[im]), "gathered")
    for x in (M, B, E, out):
        x.close()


def test_129_limbs_on_four_lanes(handle, tables):
    """4128 bits, the one size above 128 limbs that 4x37 holds: R^2 mod m comes
    from squarings there, in a context and in a plain call."""
    layout, bits, n = (4, 37, 28), 4128, 35
    m, b, e, want = _edge_case(4128, n, bits)
    tables(layout, bits, n)
    _context_powm(handle, layout, bits, m, b, e, want)
    M, B, E, out = handle.from_array(m), handle.from_array(b), handle.from_array(e), handle.integers(bits, n)
    handle.set_algorithm(xmp_amd.ALG_DISTRIBUTEDMP)
    try:
        handle.powm(out, B, E, M)
    finally:
        handle.set_algorithm(xmp_amd.ALG_DEFAULT)
    assert_rows_equal(out.get(), want, "explicit algorithm, %d bits" % bits)
    for x in (M, B, E, out):
        x.close()
