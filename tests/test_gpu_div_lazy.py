"""GPU: division by signed digits (k_div_lazy.hip), against GMP's fdiv_qr.

Every lane layout through the batch size that its rule gives it, at the largest
divisor its digits hold and one limb past the next smaller layout's, with
dividends shorter than, as long as, twice and three times the divisor.  The
edge rows: division by zero, by 1 and by powers of two, unnormalised divisors,
quotients and remainders at their extremes (a = q b and q b - 1 with q all
ones, where every digit's nearest quotient rounds up and the remainder ends
negative), and digits at the ends of the signed range."""
import numpy as np
import pytest

from helpers import O, assert_rows_equal, gmp, inputs

pytestmark = pytest.mark.gpu


def _operands(seed, n, la, lb):
    a, b = inputs.uniform(seed, n, la), inputs.uniform(seed + 1, n, lb)
    ones = np.uint32(0xFFFFFFFF)
    a[0], b[0] = ones, ones
    b[1] = 0
    b[2], b[2, 0] = 0, 1
    b[3], b[3, -1] = 0, 0x80000000
    b[4], b[4, -1], a[4] = 0, 1, ones
    b[5], b[5, lb // 2], a[5] = 0, 3, ones
    a[6] = 0
    a[7], a[7, 0] = 0, 5
    a[8], b[8] = 0xF0000000, 0x0FFFFFFF
    a[9], b[9], b[9, -1] = ones, 0, ones
    a[10], a[10, -1], b[10], b[10, -1] = 0, 0x80000000, ones, 0x7FFFFFFF
    a[11], b[11] = 0x88888888, 0x80000001
    for row, less in ((12, 0), (13, 1)):
        if la >= lb:
            d = O.to_int(b[row])
            q = (1 << 32 * (la - lb)) - 1 if la > lb else 1
            a[row] = O.from_int(q * d - less, la)
    return a, b


def _check(handle, a, b, what):
    n, la, lb = a.shape[0], a.shape[1], b.shape[1]
    zero = ~b.any(axis=1)
    wq, wr = gmp(O.GO_DIV, n, la, a, np.where(zero[:, None], np.uint32(1), b), out2_limbs=lb)
    wq[zero] = 0
    wr[zero] = np.pad(a, ((0, 0), (0, max(0, lb - la))))[zero][:, :lb]
    A, B, Q, R = handle.from_array(a), handle.from_array(b), handle.integers(32 * la, n), handle.integers(32 * lb, n)
    handle.divmod(Q, R, A, B)
    assert_rows_equal(Q.get(), wq, what + " q")
    assert_rows_equal(R.get(), wr, what + " r")
    handle.mod(R, A, B)
    assert_rows_equal(R.get(), wr, what + " mod")
    handle.div(A, A, B)   # in place
    assert_rows_equal(A.get(), wq, what + " div")
    for x in (A, B, Q, R):
        x.close()


@pytest.mark.parametrize("lb,n", [
    (9, 70), (16, 16384),                             # 4 lanes of 5 digits
    (17, 70), (24, 4096), (24, 4097), (20, 32769),    # 8x5, 4x10, 1x28
    (25, 300), (32, 4100), (32, 32770),               # 8x5, 4x10, 1x37
    (33, 33), (33, 32771), (35, 70), (34, 32769),     # 8x5, 2x19, 2x28
    (36, 17), (49, 2049), (49, 8193), (40, 16385),    # 16x5, 8x10, 4x19, 2x28
    (50, 33), (64, 2050), (64, 8200), (64, 24577),    # 16x5, 8x10, 4x19, 2x37
    (66, 14), (65, 8193),                             # 16x5, 4x19
    (67, 15), (98, 2049), (98, 8193),                 # 16x10, 8x19, 4x28
    (99, 14), (128, 2049), (129, 8193), (128, 8194),  # 16x10, 8x19, 4x37
    (130, 20), (195, 1100), (195, 8193),              # radix 2^27: 16x15, 8x29
    (196, 15), (256, 513), (256, 8193),               # 32x10, 16x19, 8x38
    (257, 14), (512, 100), (520, 2049),               # radix 2^26: 64x10, 16x40
    (521, 14), (1040, 17),                            # 64x20
])
def test_signed_digit_division(handle, lb, n):
    for la in ((2 * lb, lb + 3, lb, max(1, lb // 2), 3 * lb + 1) if n <= 300 else (2 * lb,)):
        a, b = _operands(7000 + lb + la, n, la, lb)
        _check(handle, a, b, "%d / %d limbs x %d" % (la, lb, n))


def test_signed_digit_division_long_dividends(handle):
    """Rows in LDS up to their limit, more lanes than the batch's rule gives
    where its rows would not fit, and dividends that fit none."""
    for la, lb, n in ((1024, 64, 30), (1100, 33, 4100), (3500, 20, 14), (4200, 50, 14), (9000, 300, 14)):
        a, b = _operands(7700 + la, n, la, lb)
        _check(handle, a, b, "%d / %d limbs x %d" % (la, lb, n))


def test_signed_digit_division_gathered_and_shared(handle):
    n, la, lb = 500, 96, 48
    a, b = _operands(7900, n, la, lb)
    A, B = handle.from_array(a), handle.from_array(b)
    Q, R = handle.from_array(np.zeros((n, la), np.uint32)), handle.from_array(np.zeros((n, lb), np.uint32))
    rng = np.random.Generator(np.random.PCG64(79))
    iq, ir, ia, ib = (rng.permutation(n).astype(np.uint32) for _ in range(4))
    ib[ib == 1] = 0   # row 1 is the zero divisor
    try:
        for which, idx in enumerate((iq, ir, ia, ib)):
            handle.set_indices(which, idx)
        handle.divmod(Q, R, A, B, n)
    finally:
        handle.clear_indices()
    wq, wr = gmp(O.GO_DIV, n, la, a[ia], b[ib], out2_limbs=lb)
    assert_rows_equal(Q.get()[iq], wq, "gathered q")
    assert_rows_equal(R.get()[ir], wr, "gathered r")
    one = handle.from_array(b[20:21])
    handle.divmod(Q, R, A, one, n)
    wq, wr = gmp(O.GO_DIV, n, la, a, np.repeat(b[20:21], n, axis=0), out2_limbs=lb)
    assert_rows_equal(Q.get(), wq, "shared divisor q")
    assert_rows_equal(R.get(), wr, "shared divisor r")
    for x in (A, B, Q, R, one):
        x.close()
