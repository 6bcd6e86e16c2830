"""What a batch touches of a box that has finished: nothing, until the box is detached."""
import numpy as np
import pytest

from exanbody_amd import PRECISION_FP64, Batch
from tests.helpers import RCUT, SKIN, fcc_inputs, make_pair

pytestmark = pytest.mark.gpu


def _box(seed):
    r, v, ids, L = fcc_inputs(5, temperature=1.0, seed=seed)
    _, b, _ = make_pair(r, v, ids, L)
    b.init(1.0, 1.0, RCUT, SKIN, PRECISION_FP64)
    return b


@pytest.mark.parametrize("every", [4, 0])
def test_finished_box_destroyed_before_the_others_end(every):
    """The finished box's context is destroyed without a detach (its slot stays taken); a second
    box runs on and a third is attached."""
    alone = []
    for seed, steps in ((2, 20), (3, 9)):
        b = _box(seed)
        b.run(steps, 0.004, 1.0, 1.0, RCUT, SKIN, rebuild_every=every)
        alone.append(b.export())
    batch = Batch()
    first, second, third = _box(1), _box(2), _box(3)
    q1 = batch.attach(first, 5, 0.004, 1.0, 1.0, RCUT, SKIN, rebuild_every=every)
    q2 = batch.attach(second, 20, 0.004, 1.0, 1.0, RCUT, SKIN, rebuild_every=every)
    batch.step(6)
    assert batch.status(q1) == (5, 1)
    first.close()
    spare = [_box(20 + k) for k in range(3)]  # other contexts in the memory it gave back
    batch.step(2)
    q3 = batch.attach(third, 9, 0.004, 1.0, 1.0, RCUT, SKIN, rebuild_every=every)
    while batch.step(4):
        pass
    assert batch.status(q1) == (5, 1)
    for q, b, ref in ((q2, second, alone[0]), (q3, third, alone[1])):
        batch.detach(q)
        e = b.export()
        for k in ("cell", "id", "r", "v", "f", "ep"):
            np.testing.assert_array_equal(e[k].view(np.uint8), ref[k].view(np.uint8), err_msg=k)
    batch.close()
    assert len(spare) == 3
