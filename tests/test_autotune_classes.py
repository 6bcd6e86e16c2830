"""The autotuner's shapes are cached per class; boxes that run with one and with four lanes an atom
are different classes."""
import pytest

from exanbody_amd import PRECISION_MIXED
from tests.helpers import RCUT, SKIN, fcc_inputs, make_pair

pytestmark = pytest.mark.gpu

NBH = 1  # XNB_TIMER_NBH


def test_lanes_are_part_of_the_class(monkeypatch):
    r, v, ids, L = fcc_inputs(9, rho=0.871, temperature=0.9, seed=12)
    builds = []
    for lanes in (4, 1, 4, 1):
        monkeypatch.setenv("XNB_BRICKS", f"0,0,0,{lanes}")
        _, b, _ = make_pair(r, v, ids, L)
        b.init(1.0, 1.0, RCUT, SKIN, PRECISION_MIXED)
        b.timer_enable()
        b.timer_reset()
        b.autotune(1.0, 1.0, RCUT, precision=PRECISION_MIXED)
        builds.append(b.timer_read(NBH)[1])
        b.close()
    # a class seen for the first time is timed (a build per shape), one seen before is not
    assert builds[0] > 2 and builds[1] > 2 and builds[2] == builds[3] == 1
