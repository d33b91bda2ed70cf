"""REPEAT addressing of a bilinear fetch: `wrap_pair` in csrc/image_ops.hpp takes the two
texels i and i + 1 of an axis of n texels by an addition and a compare where i lies within
one image of the origin, and by the general remainder elsewhere.  This checks the sequence
(with its unsigned 32-bit range test) against the remainder for every form: images of one
texel, both sides of each border, the ends of the 32-bit range."""
import pytest


def wrap_pair(i, n):
    m = 2 ** 32
    if (i + n) % m < 2 * n % m:
        i0 = i + n if i < 0 else i
        return i0, 0 if i0 + 1 == n else i0 + 1, True
    return i % n, (i + 1) % n, False


@pytest.mark.parametrize("n", [1, 2, 3, 16, 1279, 1920, 65535])
def test_wrap_pair_equals_the_remainder(n):
    near = set(range(-3, 4)) | {k * n + d for k in range(-3, 4) for d in range(-3, 4)}
    far = {-2 ** 31, -2 ** 31 + 1, -2 ** 31 + n, 2 ** 31 - 2, 2 ** 31 - 1 - n, 2 ** 31 - 1 - 2 * n}
    for i in near | far | set(range(-min(n, 70), min(n, 70))):
        i0, i1, fast = wrap_pair(i, n)
        assert (i0, i1) == (i % n, (i + 1) % n)
        assert fast == (-n <= i < n)
