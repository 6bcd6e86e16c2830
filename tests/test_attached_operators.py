"""Force operators called on a box while it is attached to a batch (they read the ghosts by their
slots, the batch by their sources) change nothing of what the batch computes."""
import numpy as np
import pytest

from exanbody_amd import PRECISION_FP64, PRECISION_MIXED, Batch
from tests.helpers import RCUT, SKIN, fcc_inputs, make_pair

pytestmark = pytest.mark.gpu


def _box(precision):
    r, v, ids, L = fcc_inputs(7, temperature=1.2, seed=5)
    _, b, _ = make_pair(r, v, ids, L)
    b.init(1.0, 1.0, RCUT, SKIN, precision)
    return b


@pytest.mark.parametrize("precision", [PRECISION_FP64, PRECISION_MIXED])
@pytest.mark.parametrize("lanes", [1, 4])
@pytest.mark.parametrize("every", [4, 0])
@pytest.mark.parametrize("at", [0, 2, 5])
def test_force_operator_on_an_attached_box(at, every, lanes, precision, monkeypatch):
    monkeypatch.setenv("XNB_BRICKS", f"0,0,0,{lanes}")
    a, c = _box(precision), _box(precision)
    batch = Batch()
    slot = batch.attach(a, 11, 0.004, 1.0, 1.0, RCUT, SKIN, precision=precision, rebuild_every=every)
    if at:
        batch.step(at)
    a.zero_particle_force()  # the same forces again: the first step starts from them
    a.lennard_jones_force(1.0, 1.0, RCUT, precision=precision)
    while batch.step(3):
        pass
    got = batch.detach(slot)
    batch.close()
    assert got == c.run(11, 0.004, 1.0, 1.0, RCUT, SKIN, precision=precision, rebuild_every=every)
    ea, ec = a.export(ghosts=True), c.export(ghosts=True)
    for k in ("cell", "id", "r", "v", "f", "ep"):
        np.testing.assert_array_equal(ea[k].view(np.uint8), ec[k].view(np.uint8), err_msg=k)
