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
