"""1 / sqrt(d2) as the FP64 pair loops take it (inv_sqrt_normal inside PairRange, the generic
operations outside) against IEEE's root and division, bit for bit, over its whole range."""
import numpy as np
import pytest

from tests.helpers import fcc_inputs, make_pair

pytestmark = pytest.mark.gpu


def _bits(x):
    return np.asarray(x, np.float64).view(np.uint64)


def _significands(lows):
    """Doubles of these 52 low bits under exponents over the whole range."""
    e = np.r_[1, 2, 255, 256, 257, np.arange(1000, 1047), 1500, 2020, 2021].astype(np.uint64)
    return (e[:, None] << np.uint64(52) | np.asarray(lows, np.uint64)[None, :]).ravel().view(np.float64)


def test_is_ieee():
    r, _, ids, L = fcc_inputs(4)
    _, b, _ = make_pair(r, None, ids, L)
    rng = np.random.default_rng(11)
    ones = (1 << 52) - 1
    y = rng.uniform(0.5, 2.5, 400_000)
    sq = y * y
    root = 1.0 + np.arange(1, 200_000) * 2.0 ** -52  # roots next to a power of two, from both sides
    below = 2.0 - np.arange(1, 200_000) * 2.0 ** -52
    x = np.concatenate([
        rng.uniform(1e-6, 6.25, 3_000_000),                    # squared distances within the cutoff
        np.exp2(rng.uniform(-767.0, 1000.0, 2_000_000)),       # the whole range
        np.exp2(rng.uniform(-1074.0, -760.0, 100_000)),        # below it, and its end
        sq, np.nextafter(sq, 0), np.nextafter(sq, 10),         # near the midpoints of the root
        *(f(s) for s in (root * root, below * below) for f in (lambda q: q, lambda q: np.nextafter(q, 0), lambda q: np.nextafter(q, 9))),
        # roots whose reciprocal is near a midpoint: 1 / (y + half an ulp) squared back
        1.0 / sq, np.nextafter(1.0 / sq, 0), np.nextafter(1.0 / sq, 10),
        _significands([0, 1, 2, ones, ones - 1, ones - 2, ones - 3, ones // 2, ones // 2 + 1, 0xfffffffe, 0xffffffff, 0x1fffffffe]),
        [1.0, 2.0, 4.0, 6.25, 0.25, 2.0 ** -767, np.nextafter(2.0 ** -767, 0), 2.0 ** 1000],
    ])
    x = x[(x > 0.0) & (x <= 2.0 ** 1000)]
    assert x.size > 7_000_000
    np.testing.assert_array_equal(_bits(b.fp64_inv_sqrt(x)), _bits(1.0 / np.sqrt(x)))
    b.close()
