"""GPU: divisions on both sides of the rules that choose between the signed-digit
kernels and the 32-bit ones (register, lane-pair and wave kernels), against
GMP's fdiv_qr: quotients of a few limbs, dividends shorter than the divisor, and
dividends several times the divisor in full batches.

Dividends and divisors repeat with coprime periods, so that a large batch has
1,517 different divisions, each at several places of it; among the rows division
by zero and by 1, unnormalised divisors, all-ones operands and quotients whose
digits are all ones."""
import numpy as np
import pytest

from helpers import O, gmp, inputs

pytestmark = pytest.mark.gpu

NA, NB = 37, 41


def _operands(seed, la, lb):
    a, b = inputs.uniform(seed, NA, la), inputs.uniform(seed + 1, NB, lb)
    ones = np.uint32(0xFFFFFFFF)
    b[:, -1] |= np.uint32(1)                # (a longer divisor than that is the rule)
    b[0] = 0
    b[1], b[1, 0] = 0, 1
    b[2] = ones
    b[3], b[3, -1] = 0, 0x80000000
    b[4, -1] = 0                            # a leading zero limb
    b[5, lb // 2:] = 0
    b[5, 0] |= np.uint32(1)
    b[6], b[6, -1] = 0x80000000, 0x7FFFFFFF
    a[0] = 0
    a[1] = ones
    a[2], a[2, 0] = 0, 5
    a[3], a[3, -1] = 0, 0x80000000
    if la >= lb:                            # q d - 1 and q d: the remainder at its ends
        d = O.to_int(b[7])
        q = (1 << 32 * (la - lb)) - 1 if la > lb else 1
        a[4], a[5] = O.from_int(q * d - 1, la), O.from_int(q * d, la)
        a[6, -1] = min(int(b[8, -1]), int(a[6, -1]))
    return a, b


def _assert_periodic(got, want, what):
    n, p = got.shape[0], want.shape[0]
    for k in range(0, n, p):
        part = got[k:k + p]
        bad = np.nonzero((part != want[:part.shape[0]]).any(axis=1))[0]
        assert bad.size == 0, "%s: rows %s from %d on differ" % (what, bad[:5], k)


@pytest.mark.parametrize("lb,more,n", [
    # quotients up to the rule's lengths and one limb past them
    (9, 0, 300), (15, 2, 16384), (15, 3, 300), (16, 4, 1000), (16, 5, 16384), (16, 6, 64),
    (16, -5, 300), (20, 1, 20000), (17, 4, 32768), (25, 4, 20000), (29, 5, 32768),
    (30, 2, 4097), (31, 3, 16384), (32, 7, 30000), (32, 8, 30000), (25, 2, 32769), (32, 4, 98304), (32, 5, 65536),
    (32, 10, 131073), (32, 11, 262144), (60, 6, 20000), (64, 0, 16385), (64, 7, 24576), (56, 8, 65537), (64, 9, 98304),
    (72, 3, 65536), (96, 5, 49152), (96, 6, 65536), (96, 4, 131072), (96, 12, 262144),
    (129, 4, 600), (129, 5, 16), (129, -40, 64), (130, 9, 600), (195, 10, 64), (160, 5, 2000), (160, 4, 4000),
    (196, 6, 512), (256, 7, 16), (256, 1, 1500), (384, 1, 600), (896, 1, 4096), (1040, 5, 3000), (1040, -9, 3000),
    (750, 9, 8192), (760, 5, 8192), (900, 7, 9000), (961, 3, 24577), (1016, 4, 8192), (1040, 9, 12000), (1017, 6, 11999),
    # rows that take more lanes than the batch's rule gives
    (20, 120, 65536), (24, 150, 65536), (32, 128, 65536), (32, 200, 65536), (64, 390, 65536),
    # ... and that go to the register kernels
    (24, 150, 131072), (32, 96, 131072), (40, 240, 131072), (52, 340, 131072), (64, 260, 131072),
])
def test_division_routes(handle, lb, more, n):
    la = lb + more
    a, b = _operands(9000 + lb + more, la, lb)
    rows = np.arange(min(n, NA * NB))
    x, y = a[rows % NA], b[rows % NB]
    zero = ~y.any(axis=1)
    wq, wr = gmp(O.GO_DIV, rows.size, la, x, np.where(zero[:, None], np.uint32(1), y), out2_limbs=lb)
    wq[zero] = 0
    wr[zero] = np.pad(x, ((0, 0), (0, max(0, -more))))[zero][:, :lb]
    A, B, Q, R = handle.from_array(a), handle.from_array(b), handle.integers(32 * la, n), handle.integers(32 * lb, n)
    what = "%d / %d limbs x %d" % (la, lb, n)
    handle.divmod(Q, R, A, B, n)
    _assert_periodic(Q.get(), wq, what + " q")
    _assert_periodic(R.get(), wr, what + " r")
    R.load(np.zeros((1, lb), np.uint32))
    handle.mod(R, A, B, n)
    _assert_periodic(R.get(), wr, what + " mod")
    Q.load(np.zeros((1, la), np.uint32))
    handle.div(Q, A, B, n)
    _assert_periodic(Q.get(), wq, what + " div")
    for z in (A, B, Q, R):
        z.close()


@pytest.mark.parametrize("lb,la,n", [
    (9, 8, 300), (17, 16, 70), (24, 1, 4097), (32, 30, 40000), (35, 34, 33), (49, 47, 7826), (64, 32, 30000), (98, 97, 9000),
    (129, 64, 700), (195, 194, 9), (256, 1, 600), (401, 399, 70), (520, 519, 2100), (831, 829, 65),
])
def test_dividends_of_fewer_limbs(handle, lb, la, n):
    """Divisors that are all longer than the dividends, and batches with one that
    is not at its start, within or at its end: a shorter one, 1 and 0."""
    a, b = inputs.uniform(9300 + lb, n, la), inputs.uniform(9301 + lb, n, lb)
    b[:, -1] |= np.uint32(1)
    b[2 % n, la:], b[2 % n, la] = 0, 1                  # one bit more than the dividends have
    A, Q, R = handle.from_array(a), handle.integers(32 * la, n), handle.integers(32 * lb, n)
    for at in (None, 0, n // 2, n - 1):
        for d in ([None] if at is None else [O.to_int(a[at]) >> 1, O.to_int(a[at]), 1, 0]):
            c = b.copy()
            if d is not None:
                c[at] = O.from_int(d, lb)
            B = handle.from_array(c)
            handle.divmod(Q, R, A, B)
            wq, wr = np.zeros_like(a), np.pad(a, ((0, 0), (0, lb - la)))
            if d:
                x = O.to_int(a[at])
                wq[at], wr[at] = O.from_int(x // d, la), O.from_int(x % d, lb)
            what = "%d / %d limbs x %d, %s at %s" % (la, lb, n, d if d is None or d < 2 else "a short one", at)
            _assert_periodic(Q.get(), wq, what + " q")
            _assert_periodic(R.get(), wr, what + " r")
            B.close()
    for x in (A, Q, R):
        x.close()


@pytest.mark.parametrize("lb,la,n", [
    (17, 271, 24576), (24, 272, 33000), (20, 192, 33001), (24, 143, 50001), (17, 144, 66000), (25, 150, 66001),
    (32, 256, 24576), (33, 288, 30000), (48, 320, 40000), (49, 168, 50001), (64, 192, 66001), (65, 384, 24576),
    (96, 192, 50001), (96, 288, 66001), (97, 448, 24576), (128, 447, 24576),
    (24, 72, 131072), (32, 47, 131072), (48, 72, 150000), (64, 96, 131072), (96, 143, 131072), (128, 192, 131072),
])
def test_gathered_long_dividends(handle, lb, la, n):
    """Both sides of the rule for dividends that an index array gathers, and the
    same sizes without one."""
    a, b = _operands(9400 + lb + la, la, lb)
    rows = np.arange(NA * NB)
    x, y = a[rows % NA], b[rows // NA]
    zero = ~y.any(axis=1)
    wq, wr = gmp(O.GO_DIV, rows.size, la, x, np.where(zero[:, None], np.uint32(1), y), out2_limbs=lb)
    wq[zero], wr[zero] = 0, x[zero][:, :lb]
    rng = np.random.default_rng(la)
    ia, ib = rng.integers(0, NA, n).astype(np.uint32), rng.integers(0, NB, n).astype(np.uint32)
    A, B, Q, R = handle.from_array(a), handle.from_array(b), handle.integers(32 * la, n), handle.integers(32 * lb, n)
    what = "%d / %d limbs x %d" % (la, lb, n)
    handle.set_indices(2, ia)
    handle.set_indices(3, ib)
    try:
        handle.divmod(Q, R, A, B, n)
    finally:
        handle.clear_indices()
    pair = ia.astype(np.int64) + NA * ib
    assert np.array_equal(Q.get(), wq[pair]), what + " gathered q"
    assert np.array_equal(R.get(), wr[pair]), what + " gathered r"
    handle.divmod(Q, R, A, B, n)
    pair = np.arange(n) % NA + NA * (np.arange(n) % NB)
    assert np.array_equal(Q.get(), wq[pair]), what + " q"
    assert np.array_equal(R.get(), wr[pair]), what + " r"
    for z in (A, B, Q, R):
        z.close()


@pytest.mark.parametrize("lb,la,n,stored", [
    (24, 320, 50001, True), (17, 240, 66001, False), (28, 600, 24576, True), (32, 384, 131071, False), (40, 480, 66000, True),
    (48, 576, 66001, True), (56, 448, 50001, False), (64, 384, 66001, True), (80, 768, 33001, True), (96, 576, 50001, False),
])
def test_long_dividends_of_middling_batches(handle, lb, la, n, stored):
    """The first dividends that go to the lane pairs, and one limb less."""
    for la in (la - 1, la):
        a, b = _operands(9500 + lb + la, la, lb)
        rows = np.arange(NA * NB)
        x, y = a[rows % NA], b[rows % NB]
        zero = ~y.any(axis=1)
        wq, wr = gmp(O.GO_DIV, rows.size, la, x, np.where(zero[:, None], np.uint32(1), y), out2_limbs=lb)
        wq[zero], wr[zero] = 0, x[zero][:, :lb]
        A, B, Q, R = handle.from_array(a), handle.from_array(b), handle.integers(32 * la, n), handle.integers(32 * lb, n)
        what = "%d / %d limbs x %d" % (la, lb, n)
        if stored:
            handle.divmod(Q, R, A, B, n)
            _assert_periodic(Q.get(), wq, what + " q")
        else:
            handle.mod(R, A, B, n)
        _assert_periodic(R.get(), wr, what + " r")
        for z in (A, B, Q, R):
            z.close()
