"""GPU: products on the matrix cores (k_mul_mx.hip) and Karatsuba above them,
against GMP's mpz_mul.

Sizes on both sides of the kernel's edges: operands that end inside, at and
past a 16-byte block, products that end inside and at a 256-digit tile and a
group of tiles, multipliers down to one limb, truncated and padded outputs;
batches whose last workgroup holds one product of two; squares, index arrays,
a shared multiplier, in place.  The edge rows put every balanced digit at its
extremes and run a carry through a whole operand."""
import numpy as np
import pytest

from helpers import O, assert_rows_equal, gmp, inputs

pytestmark = pytest.mark.gpu


def _pair(seed, n, la, lb):
    a, b = inputs.uniform(seed, n, la), inputs.uniform(seed + 1, n, lb)
    if n >= 8:
        a[0], b[0] = 0xFFFFFFFF, 0xFFFFFFFF
        a[1], a[1, 0], b[1] = 0x7F7F7F7F, 0x80808080, 0x7F7F7F7F   # the carry of limb 0 crosses every limb
        a[2], b[2] = 0x7F7F7F7F, 0x80808080
        a[3], b[3] = 0, 0xFFFFFFFF
        a[4], b[4] = 0x80808080, 0x7F7F7F80
        a[5] = 0
        a[5, -1] = 0x80000000
        a[6], b[6], b[6, 0] = 0xFFFFFFFF, 0, 1                      # digits -1: a borrow under every limb
        a[7], b[7] = 0x80000000, 0x00000001
    return a, b


@pytest.mark.parametrize("la,lb,lp,n", [
    (17, 17, 34, 9),          # one tile, one product a workgroup
    (32, 17, 49, 300),
    (33, 20, 53, 8),          # a multiplier that ends at a block
    (63, 63, 126, 65),
    (64, 64, 128, 9),         # 128 limbs: whole tiles
    (64, 64, 100, 9),         # truncated inside a tile
    (65, 64, 140, 9),         # padded past the product
    (128, 127, 255, 600),     # two products a workgroup
    (128, 128, 256, 513),     # ... and one in the last
    (130, 67, 197, 8),
    (255, 130, 300, 515),     # truncated at two products a workgroup
    (512, 256, 768, 9),
    (512, 512, 1024, 513),
    (513, 1, 514, 9),         # the shortest multiplier
    (515, 3, 518, 520),       # eight tiles at a time
    (1024, 1024, 2048, 513),
    (1000, 1023, 2100, 514),
    (1025, 1000, 2025, 9),    # beyond: one product, four tiles at a time
    (2048, 2048, 4096, 9),    # the largest the kernel holds
    (3000, 1096, 4096, 8),
    (2049, 2048, 4097, 9),    # one limb more: Karatsuba, its halves on the matrix cores
    (4100, 2050, 6150, 8),
    (4096, 30, 4126, 8),      # a alone is split
])
def test_matrix_core_products(handle, la, lb, lp, n):
    a, b = _pair(6100 + la + lb, n, la, lb)
    A, B, P = handle.from_array(a), handle.from_array(b), handle.integers(32 * lp, n)
    handle.mul(P, A, B)
    want = gmp(O.GO_MUL, n, lp, a, b)
    assert_rows_equal(P.get(), want, "%d x %d -> %d limbs" % (la, lb, lp))
    handle.mul(P, B, A)
    assert_rows_equal(P.get(), want, "%d x %d -> %d limbs, swapped" % (la, lb, lp))
    if lp >= 2 * la:
        handle.mul(P, A, A)
        assert_rows_equal(P.get(), gmp(O.GO_MUL, n, lp, a, a), "square of %d limbs" % la)
    for x in (A, B, P):
        x.close()


@pytest.mark.parametrize("limbs,n", [(40, 77), (128, 777), (600, 515)])
def test_matrix_core_products_gathered_shared_in_place(handle, limbs, n):
    a, b = _pair(6300 + limbs, n, limbs, limbs)
    A, B, P = handle.from_array(a), handle.from_array(b), handle.from_array(np.zeros((n, 2 * limbs), np.uint32))
    rng = np.random.Generator(np.random.PCG64(63))
    ip, ia, ib = (rng.permutation(n).astype(np.uint32) for _ in range(3))
    try:
        for which, idx in enumerate((ip, ia, ib)):
            handle.set_indices(which, idx)
        handle.mul(P, A, B, n)
    finally:
        handle.clear_indices()
    want = np.zeros((n, 2 * limbs), np.uint32)
    want[ip] = gmp(O.GO_MUL, n, 2 * limbs, a[ia], b[ib])
    assert_rows_equal(P.get(), want, "gathered")
    one = handle.from_array(b[:1])
    handle.mul(P, A, one, n)
    assert_rows_equal(P.get(), gmp(O.GO_MUL, n, 2 * limbs, a, np.repeat(b[:1], n, axis=0)), "a shared multiplier")
    handle.mul(A, A, B, n)
    assert_rows_equal(A.get(), gmp(O.GO_MUL, n, limbs, a, b), "in place, truncated")
    for x in (A, B, P, one):
        x.close()


def test_beyond_the_matrix_cores(fresh_handle):
    """One limb past what the kernel holds: all-ones operands through
    Karatsuba's carry terms, and the schoolbook where the scratch limit leaves
    Karatsuba no room."""
    h, n, limbs = fresh_handle, 3, 2049
    ones = np.full((n, limbs), 0xFFFFFFFF, np.uint32)
    a, b = _pair(6500, n, limbs, limbs)
    A, B, S, P = h.from_array(ones), h.from_array(b), h.from_array(a), h.integers(64 * limbs, n)
    for limit in (0, 4096):
        h.set_scratch_limit(limit)
        h.mul(P, A, A)
        assert_rows_equal(_get(h, P), gmp(O.GO_MUL, n, 2 * limbs, ones, ones), "all ones, limit %d" % limit)
        h.set_scratch_limit(limit)
        h.mul(P, S, B)
        assert_rows_equal(_get(h, P), gmp(O.GO_MUL, n, 2 * limbs, a, b), "limit %d" % limit)
    for x in (A, B, S, P):
        x.close()


def _get(h, x):
    h.set_scratch_limit(0)   # the export's staging is scratch too
    return x.get()


@pytest.mark.parametrize("limbs", [17, 20, 25, 28, 32])
@pytest.mark.parametrize("n", [1, 1000, 2049])
def test_truncated_products_on_both_kernels(handle, limbs, n):
    """Products and squares whose last limb asked for is at the lines between
    the lane kernels and the matrix cores."""
    a, b = inputs.uniform(5600 + limbs, n, limbs), inputs.uniform(5700 + limbs, n, limbs)
    a[0], b[0] = 0xFFFFFFFF, 0xFFFFFFFF
    A, B = handle.from_array(a), handle.from_array(b)
    for lp in sorted({limbs, 25, 26, 36, 37, 2 * limbs, 2 * limbs + 3}):
        if lp < limbs:
            continue
        P = handle.integers(32 * lp, n)
        handle.mul(P, A, B)
        assert_rows_equal(P.get(), gmp(O.GO_MUL, n, lp, a, b), "%d x %d -> %d limbs" % (limbs, limbs, lp))
        handle.mul(P, A, A)
        assert_rows_equal(P.get(), gmp(O.GO_MUL, n, lp, a, a), "%d limbs squared -> %d" % (limbs, lp))
        P.close()
    for x in (A, B):
        x.close()
