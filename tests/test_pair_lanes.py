"""What the fast FP64 pair hands over to the generic operations, with one lane and with four lanes
an atom, against the oracle's IEEE operations bit for bit.  The pairs stand alone, some of them
within the list's radius but beyond the cutoff: there the fast pair adds 0 * infinity for
eps 1e308, where the generic one adds nothing."""
import numpy as np
import pytest

from tests.test_fp64_pair_range import _compare, _near, _rows

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True, params=[1, 4])
def lanes(request, monkeypatch):
    monkeypatch.setenv("XNB_BRICKS", f"0,0,0,{request.param}")
    return request.param


@pytest.mark.parametrize("eps,sigma", [(1e308, 1.0), (-1e308, 0.9), (np.inf, 1.0), (np.nan, 1.0), (1.0, 1e31), (1.0, 2.0 ** 100),
                                       (1.0, 1e120), (1.0, np.nan), (0.0, 1.0)])
def test_parameters(eps, sigma):
    dx = np.random.default_rng(6).uniform(0.7, 2.75, 600)
    ge = _compare(*_rows(dx), eps=eps, sigma=sigma)
    beyond = np.repeat(dx > 2.5, 2)
    assert beyond.sum() > 50
    f = np.empty_like(ge["f"])
    f[ge["id"].astype(np.int64)] = ge["f"]
    assert np.all(f[beyond] == 0.0)


@pytest.mark.parametrize("sigma", [1e-120, 1e-3, 1.0])
def test_distances(sigma):
    """Coincident atoms, squared distances below 2^-767, and roots next to powers of two."""
    dx = [0.0, 1e-200, 1e-162, 1e-140, 8e-116, 2e-115, 1e-30, 0.5, 2.4]
    dx += [d for k in range(-4, 2) for d in _near(2.0 ** k, 6)]
    _compare(*_rows(np.array(dx)), sigma=sigma)
