"""The plain FP64 pair loop's fast root and reciprocal (inv_sqrt_normal) against the oracle's
IEEE operations, bit for bit, where the fast sequence has to hand over to the generic ones:
roots whose significand is all ones, coincident and near-coincident atoms, and parameters it
does not cover; and at the edges of its range."""
import numpy as np
import pytest

from exanbody_amd import PRECISION_FP64
from tests.helpers import RCUT, make_pair

pytestmark = pytest.mark.gpu


def _rows(dx):
    """One pair per row, a at x = 0 and b at x = dx exactly, rows 3 apart (beyond the cutoff)."""
    m = int(np.ceil(np.sqrt(len(dx))))
    k = np.arange(len(dx))
    a = np.stack([np.zeros(len(dx)), 3.0 * (k % m), 3.0 * (k // m)], axis=1)
    b = a.copy()
    b[:, 0] = dx
    r = np.empty((2 * len(dx), 3))
    r[0::2], r[1::2] = a, b
    return r, 3.0 * m


def _compare(r, L, eps=1.0, sigma=1.0, rcut=RCUT):
    ids = np.arange(len(r), dtype=np.uint64)
    o, b, _ = make_pair(r, None, ids, L)
    o.init(1.0, 1.0, RCUT, 0.3)
    b.init(1.0, 1.0, RCUT, 0.3, PRECISION_FP64)
    for x in (o, b):
        getattr(x, "zero_force" if x is o else "zero_particle_force")()
    with np.errstate(all="ignore"):
        o.lj_force(eps, sigma, rcut)
    b.lennard_jones_force(eps, sigma, rcut, precision=PRECISION_FP64)
    oe, ge = o.export(), b.export()
    np.testing.assert_array_equal(oe["id"], ge["id"])
    for k in ("f", "ep"):
        assert np.array_equal(np.isnan(oe[k]), np.isnan(ge[k])), k
        ok = ~np.isnan(oe[k])
        np.testing.assert_array_equal(oe[k][ok].view(np.uint64), ge[k][ok].view(np.uint64), err_msg=k)
    return ge


def _near(x, steps):
    out, y = [x], x
    for _ in range(steps):
        y = np.nextafter(y, 0.0)
        out.append(y)
    y = x
    for _ in range(steps):
        y = np.nextafter(y, 10.0)
        out.append(y)
    return out


def test_roots_next_to_powers_of_two():
    """dx and the values next to it for dx = 2^k: among them every root with an all-ones
    significand between 2^-9 and 2.5 (sqrt(RN(dx^2)) = dx)."""
    dx = np.array([d for k in range(-9, 2) for d in _near(2.0 ** k, 20)])
    dx = dx[dx < RCUT]
    ones = dx.view(np.uint64) & np.uint64((1 << 52) - 1) == np.uint64((1 << 52) - 1)
    assert ones.sum() >= 10
    ge = _compare(*_rows(dx))
    assert np.all(ge["f"][:, 0] != 0.0)  # every pair was found (the energy is 0 at dx = sigma)
    _compare(*_rows(dx), eps=0.37, sigma=0.011)


def test_random_distances():
    rng = np.random.default_rng(3)
    r, L = _rows(rng.uniform(0.7, 2.6, 20000))
    _compare(r, L)
    _compare(r, L, eps=0.37, sigma=1.13, rcut=2.25)


def test_cutoff_sphere():
    """d2 on both sides of rc^2, by one unit in the last place."""
    ge = _compare(*_rows(np.array(_near(RCUT, 8))))
    assert (ge["ep"] != 0.0).any() and (ge["ep"] == 0.0).any()


@pytest.mark.parametrize("sigma", [1e-120, 1e-116, 1e-3])
def test_coincident_and_tiny_distances(sigma):
    """Distances from 0 through d2 < 2^-767 (the fast range's end) to normal ones in one box."""
    dx = np.array([0.0, 1e-200, 1e-162, 1e-155, 1e-140, 3e-116, 8e-116, 2e-115, 1e-100, 1e-30, 1e-3, 0.5, 1.0, 2.4])
    _compare(*_rows(dx), sigma=sigma)


@pytest.mark.parametrize("eps,sigma", [(1e308, 1.0), (np.inf, 1.0), (np.nan, 1.0), (1.0, 1e31), (1.0, 2.0 ** 100), (1.0, np.nan),
                                       (0.0, 1.0), (-1.0, 0.9), (1.0, 0.0)])
def test_parameters(eps, sigma):
    rng = np.random.default_rng(4)
    _compare(*_rows(rng.uniform(0.7, 2.6, 500)), eps=eps, sigma=sigma)
