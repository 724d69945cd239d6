"""GPU: exponentiation on the matrix cores (k_powm_mx.hip), against GMP.

Every block count that is compiled, at its widest size and at the smallest
that takes it (where the top blocks hold no digits), with moduli, bases and
exponents at the edges of the balanced-digit representation: all ones, 1, 3, the
top bit alone, leading zero limbs, bases above the modulus, digits at +127
and -128, even and zero moduli.  One batch is long enough for the carries that
the fast path leaves to its rounds."""
import numpy as np
import pytest

from helpers import O, assert_rows_equal, gmp, inputs

pytestmark = pytest.mark.gpu

# widest sizes of the compiled block counts, and one limb above the next smaller
SIZES = [512, 1024, 1536, 2048, 2560, 3072, 3584, 4096, 5120, 6144, 7168, 8192]
SIZES += [160, 256, 288] + [b + 32 for b in SIZES[:-1]]


def _edge_rows(m, b, e):
    ones = np.uint32(0xFFFFFFFF)
    m[0], b[0], b[0, 0], e[0] = ones, ones, ones - 1, ones          # 2^bits - 1, base m - 1
    m[1] = 0
    m[1, 0] = 1                                                     # m = 1
    m[2] = 0
    m[2, 0], b[2] = 3, ones                                         # a base far above the modulus
    m[3] = 0
    m[3, 0], m[3, -1], b[3] = 1, 0x80000000, ones                   # 2^(bits-1) + 1
    m[4, -1], b[4] = 0, ones                                        # a leading zero limb
    e[5] = 0
    b[6] = 0
    m[7], b[7] = 0x7F7F7F7F, 0x80808080                             # digits at +127, and at -128 with carries
    m[8], b[8] = 0x80808080, 0x7F7F7F7F
    m[8, 0] = 0x80808081
    m[9], m[9, 0], m[9, -1] = 0x80808080, 0x80808081, 0x7F7F7F7F    # just below R/2 in balanced digits
    m[10, 0] &= ones - 1                                            # even
    m[11] = 0


@pytest.mark.parametrize("bits", sorted(SIZES))
def test_matrix_core_powm_edges(handle, bits):
    n, exp_bits = 14, 96
    m, b, e = inputs.powm_class(4100 + bits, n, bits, exp_bits=exp_bits)
    _edge_rows(m, b, e)
    want = np.zeros_like(m)
    odd = (m[:, 0] & 1).astype(bool)
    want[odd] = gmp(O.GO_POWM, int(odd.sum()), bits // 32, b[odd], e[odd], m[odd])
    M, B, E = handle.from_array(m), handle.from_array(b), handle.from_array(e)
    out = handle.integers(bits, n)
    handle.powm(out, B, E, M)
    assert_rows_equal(out.get(), want, "%d bits" % bits)
    # in place
    handle.powm(B, B, E, M)
    assert_rows_equal(B.get(), want, "%d bits in place" % bits)
    for x in (M, B, E, out):
        x.close()


@pytest.mark.parametrize("bits", [5152, 6144, 6176, 7168, 7200, 8192])
def test_matrix_core_powm_crowded(handle, bits):
    """More instances than SIMDs: moduli above 5120 bits keep m' in LDS."""
    n = 1030
    m, b, e = inputs.powm_class(4700 + bits, n, bits, exp_bits=32)
    _edge_rows(m, b, e)
    want = np.zeros_like(m)
    odd = (m[:, 0] & 1).astype(bool)
    want[odd] = gmp(O.GO_POWM, int(odd.sum()), bits // 32, b[odd], e[odd], m[odd])
    M, B, E = handle.from_array(m), handle.from_array(b), handle.from_array(e)
    out = handle.integers(bits, n)
    handle.powm(out, B, E, M)
    assert_rows_equal(out.get(), want, "%d bits" % bits)
    for x in (M, B, E, out):
        x.close()


@pytest.mark.parametrize("bits,count", [(480, 2048), (512, 2048), (640, 3072), (1024, 4096), (2048, 4096), (4096, 512)])
def test_matrix_core_powm_long_runs(handle, bits, count):
    """Batches of full-length exponents: millions of limb sums, some of whose
    moved high words carry (about one limb in 2^15) and some of whose top
    limbs do (and m is subtracted once more)."""
    m, b, e = inputs.powm_class(4500 + bits, count, bits)
    M, B, E = handle.from_array(m), handle.from_array(b), handle.from_array(e)
    out = handle.integers(bits, count)
    handle.powm(out, B, E, M)
    assert_rows_equal(out.get(), gmp(O.GO_POWM, count, bits // 32, b, e, m), "%d x %d bits" % (count, bits))
    for x in (M, B, E, out):
        x.close()


def test_matrix_core_powm_gathered_and_shared(handle):
    """Index arrays on every operand, a modulus and an exponent shared by all,
    and exponents shorter and longer than the modulus."""
    bits, n = 2048, 200
    m, b, e = inputs.powm_class(4900, n, bits)
    rng = np.random.Generator(np.random.PCG64(49))
    io, ib, ie, im = (rng.permutation(n).astype(np.uint32) for _ in range(4))
    M, B, E = handle.from_array(m), handle.from_array(b), handle.from_array(e)
    out = handle.from_array(np.zeros_like(m))
    try:
        for which, idx in enumerate((io, ib, ie, im)):
            handle.set_indices(which, idx)
        handle.powm(out, B, E, M, n)
    finally:
        handle.clear_indices()
    want = np.zeros_like(m)
    want[io] = gmp(O.GO_POWM, n, bits // 32, b[ib], e[ie], m[im])
    assert_rows_equal(out.get(), want, "gathered")
    for exp_bits in (32, 2048 + 64):
        e1 = inputs.uniform(4901, 1, exp_bits // 32)
        M1, E1 = handle.from_array(m[:1]), handle.from_array(e1)
        handle.powm(out, B, E1, M1, n)
        want = gmp(O.GO_POWM, n, bits // 32, b, np.repeat(e1, n, axis=0), np.repeat(m[:1], n, axis=0))
        assert_rows_equal(out.get(), want, "shared modulus, %d-bit exponent" % exp_bits)
        M1.close()
        E1.close()
    for x in (M, B, E, out):
        x.close()


@pytest.mark.parametrize("counts", [(30, 20, 10, 5), (9000, 4000, 300, 3), (12500, 0, 0, 2)])
def test_batch_of_matrix_core_and_queued_classes(handle, counts):
    """A mixed batch whose classes all run on the matrix cores, one whose short
    moduli go to the queue (the classes share the GPU, so the rule sees the
    whole batch), and one with a single class of each; replayed on new inputs."""
    from xmp_amd import ext

    sizes = [bits for bits, c in zip((512, 1024, 3072, 4096), counts) if c]
    counts = [c for c in counts if c]
    arrays = [[handle.integers(b, c) for _ in range(2)] + [handle.integers(96, c), handle.integers(b, c)]
              for b, c in zip(sizes, counts)]
    batch = None
    for seed in (1, 2, 3):
        wants = []
        for (out, B, E, M), bits, c in zip(arrays, sizes, counts):
            m, b, e = inputs.powm_class(5000 + 10 * seed + bits, c, bits, exp_bits=96)
            for x, v in ((M, m), (B, b), (E, e)):
                x.load(v)
            wants.append(gmp(O.GO_POWM, c, bits // 32, b, e, m))
        if batch is None:
            batch = ext.Batch(handle, *[[a[k] for a in arrays] for k in range(4)], counts)
        else:
            batch.prepare()
        batch.launch_async()
        for (out, _, _, _), want, bits in zip(arrays, wants, sizes):
            assert_rows_equal(out.get(), want, "launch %d, %d bits" % (seed, bits))
    batch.close()
    for a in arrays:
        for x in a:
            x.close()
