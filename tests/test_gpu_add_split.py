"""GPU: sums and differences of batches whose limbs are split over the waves of a
workgroup, against Python integers: lengths at the edges of a wave's chunk (8
and 16 limbs) and of one pass (128 and 256), shorter operands, carries and
borrows that run through whole chunks and through all of them, batches that
end inside a row of 64, in place."""
import numpy as np
import pytest

from helpers import inputs

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (7, 8, 8), (8, 8, 9), (9, 5, 10), (64, 3, 64), (127, 128, 128), (128, 128, 129), (1, 256, 256),
          (256, 256, 257), (300, 700, 1000)]


def _ints(x):
    return [int.from_bytes(r.tobytes(), "little") for r in x]


@pytest.mark.parametrize("la,lb,ls", SHAPES)
@pytest.mark.parametrize("n", [1, 63, 131])
def test_split_add_sub(handle, la, lb, ls, n):
    a, b = inputs.uniform(9100 + la + n, n, la), inputs.uniform(9200 + lb + n, n, lb)
    ones = np.uint32(0xFFFFFFFF)
    a[0::9], b[0::9] = ones, 0
    b[0::9, 0] = 1                          # a carry through everything
    a[1::9], b[1::9] = 0, 0
    b[1::9, 0] = 1                          # a borrow through everything
    a[2::9, 1:], b[2::9, 1:] = ones, 0      # a carry, if the first limbs give one
    a[3::9, 8:16], b[3::9, 8:16] = ones, 0  # chunks that pass a carry on
    a[4::9, 16:32], b[4::9, 16:32] = 0, 0   # or a borrow
    a[5::9], b[5::9] = ones, ones
    mod = 1 << (32 * ls)
    ia, ib = _ints(a), _ints(b)
    A, B, S = handle.from_array(a), handle.from_array(b), handle.integers(32 * ls, n)
    handle.add(S, A, B)
    assert _ints(S.get()) == [(x + y) % mod for x, y in zip(ia, ib)]
    handle.sub(S, A, B)
    assert _ints(S.get()) == [(x - y) % mod for x, y in zip(ia, ib)]
    if la == ls:
        handle.sub(A, A, B)
        assert _ints(A.get()) == [(x - y) % mod for x, y in zip(ia, ib)]
    for x in (A, B, S):
        x.close()


def test_both_sides_of_the_split(handle):
    """The largest split batch and the next one agree."""
    a, b = inputs.uniform(9300, 196609, 19), inputs.uniform(9301, 196609, 17)
    out = []
    for n in (196608, 196609):
        A, B, S = handle.from_array(a[:n]), handle.from_array(b[:n]), handle.integers(32 * 20, n)
        handle.add(S, A, B)
        out.append(S.get())
        handle.sub(S, A, B)
        out.append(S.get())
        for x in (A, B, S):
            x.close()
    assert np.array_equal(out[0], out[2][:-1])
    assert np.array_equal(out[1], out[3][:-1])
