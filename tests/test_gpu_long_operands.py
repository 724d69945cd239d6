"""GPU: the kernels behind the matrix-core products and the signed-digit
divisions, against GMP: Karatsuba (more than 4,096 limbs in all, and the
schoolbook where no workspace is allowed), one wave a division (divisors of
more than 1,040 limbs), lane pairs and registers (short quotients in the
batches that go to them, dividends too long for rows in LDS).

Karatsuba's cases walk the split's branches: both operands split, the longer
alone, two levels, truncated and padded outputs, all-ones operands, the one
term past the product (ca cb B^2 at limb 3h = len(a) + len(b)) with the
product's end on a chunk boundary, squares, index arrays with a shared
multiplier, in place.  The divisions' are the operands whose estimate is one
too large, limbs at the carry and borrow extremes, unnormalised divisors and
zero."""
import numpy as np
import pytest

from helpers import O, assert_rows_equal, gmp, inputs
from test_gpu_arith import _addback_cases, _later_digit_cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("la,lb,lp", [
    (2050, 2050, 4100),    # both split
    (2751, 1377, 4160),    # 3h = 4128 limbs, 258 chunks of 16
    (4500, 600, 5100),     # the longer one alone
    (4100, 4098, 8198),    # two levels
    (2100, 2050, 2200),    # truncated
    (2100, 2050, 4300),    # wider than the product
])
def test_karatsuba_products(handle, la, lb, lp):
    n = 67
    a, b = inputs.uniform(9500 + la, n, la), inputs.uniform(9501 + lb, n, lb)
    a[0], b[0] = 0xFFFFFFFF, 0xFFFFFFFF
    b[1] = 0
    a[2, la // 2:] = 0xFFFFFFFF
    A, B, P = handle.from_array(a), handle.from_array(b), handle.integers(32 * lp, n)
    want = gmp(O.GO_MUL, n, lp, a, b)
    handle.mul(P, A, B)
    assert_rows_equal(P.get(), want, "%d x %d -> %d limbs" % (la, lb, lp))
    handle.mul(P, B, A)
    assert_rows_equal(P.get(), want, "%d x %d -> %d limbs, swapped" % (la, lb, lp))
    if lp >= 2 * la:
        handle.mul(P, A, A)
        assert_rows_equal(P.get(), gmp(O.GO_MUL, n, lp, a, a), "%d limbs squared" % la)
    for x in (A, B, P):
        x.close()


def test_karatsuba_indices_shared_and_in_place(handle):
    n, limbs = 70, 2100
    a, b = inputs.uniform(9600, n, limbs), inputs.uniform(9601, 3, limbs)
    rng = np.random.default_rng(96)
    ia, ip = rng.permutation(n).astype(np.uint32), rng.permutation(n).astype(np.uint32)
    A, B, P = handle.from_array(a), handle.from_array(b), handle.integers(64 * limbs, n)
    handle.set_indices(0, ip)
    handle.set_indices(1, ia)
    try:
        handle.mul(P, A, B)
    finally:
        handle.clear_indices()
    assert_rows_equal(P.get()[ip], gmp(O.GO_MUL, n, 2 * limbs, a[ia], b[np.arange(n) % 3]), "indexed")
    handle.mul(A, A, A)
    assert_rows_equal(A.get(), gmp(O.GO_MUL, n, limbs, a, a), "square in place")
    for x in (A, B, P):
        x.close()


def test_schoolbook_without_a_workspace(fresh_handle):
    h, n, la, lb = fresh_handle, 40, 4100, 30
    a, b = inputs.uniform(9700, n, la), inputs.uniform(9701, n, lb)
    A, B, P = h.from_array(a), h.from_array(b), h.integers(32 * (la + lb), n)
    h.set_scratch_limit(4096)
    try:
        h.mul(P, A, B)
    finally:
        h.set_scratch_limit(0)
    assert_rows_equal(P.get(), gmp(O.GO_MUL, n, la + lb, a, b), "schoolbook")
    for x in (A, B, P):
        x.close()


def _check(handle, a, b, n, what):
    """n divisions of the repeated operands; every row compared."""
    rows, la, lb = a.shape[0], a.shape[1], b.shape[1]
    zero = ~b.any(axis=1)
    wq, wr = gmp(O.GO_DIV, rows, la, a, np.where(zero[:, None], np.uint32(1), b), out2_limbs=lb)
    wq[zero] = 0
    wr[zero] = a[zero][:, :lb]
    A, B, Q, R = handle.from_array(a), handle.from_array(b), handle.integers(32 * la, n), handle.integers(32 * lb, n)
    handle.divmod(Q, R, A, B, n)
    q, r = Q.get(), R.get()
    for k in range(0, n, rows):
        assert_rows_equal(q[k:k + rows], wq[:min(rows, n - k)], what + " q")
        assert_rows_equal(r[k:k + rows], wr[:min(rows, n - k)], what + " r")
    for x in (A, B, Q, R):
        x.close()


# (divisor's limbs, divisions, limbs that the dividends are moved up by): one
# wave each, lane pairs, registers
@pytest.mark.parametrize("nb,n,up", [
    (130, 384, 0), (195, 384, 0), (1041, 100, 0), (1100, 60, 40),
    (32, 17000, 0), (64, 17000, 0), (96, 50000, 0), (128, 60, 3700), (50, 60, 4200),
    (16, 17000, 0), (16, 17000, 9), (9, 20000, 3), (96, 131072, 0), (32, 131073, 0),
])
def test_estimates_one_too_large(handle, nb, n, up):
    k = min(n, 384)
    for what, (a, b) in (("add-back", _addback_cases(nb, k, 9800 + nb)),
                         ("later digits", _later_digit_cases(nb, k, 9900 + nb))):
        a = np.pad(a, ((0, 0), (up, 0)))
        _check(handle, a, b, n, "%s, %d limbs x %d" % (what, nb, n))


@pytest.mark.parametrize("la,lb,n", [(1341, 1041, 70), (2300, 1130, 40), (3800, 130, 60), (3900, 128, 60), (48, 16, 17000)])
def test_divisions_at_the_carries(handle, la, lb, n):
    k = min(n, 300)
    rng = np.random.default_rng(99)
    vals = np.array([0, 1, 0x7FFFFFFF, 0x80000000, 0xFFFFFFFE, 0xFFFFFFFF], np.uint32)
    a, b = vals[rng.integers(0, len(vals), (k, la))], vals[rng.integers(0, len(vals), (k, lb))]
    b[:, -1] |= np.uint32(0x80000000)
    a[0], b[0] = 0xFFFFFFFF, 0xFFFFFFFF
    a[1], b[1], b[1, -1] = 0xFFFFFFFF, 0, 0x80000000
    b[2] = 0
    b[3], b[3, 0] = 0, 1
    a[4, lb:] = 0
    for i in range(5, 25):   # unnormalised
        top = int(rng.integers(1, lb + 1))
        b[i, top:] = 0
        b[i, top - 1] = (int(b[i, top - 1]) >> int(rng.integers(0, 32))) | 1
    _check(handle, a, b, n, "%d / %d limbs x %d" % (la, lb, n))
