"""Boxes on both sides of the bounds that decide which boxes of a batch take four lanes an atom
(their own atoms and the batch's, by kind of rebuild), in one batch, against the same boxes run
alone, bit for bit."""
import numpy as np
import pytest

from exanbody_amd import PRECISION_FP64, PRECISION_MIXED, Batch
from tests.test_batch_quads import RCUT, SKIN, box

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("every,sizes", [
    # more than 98,304 atoms from the fourth box on
    (0, (60000, 8192, 8193, 30000, 8192, 4096, 4097)),
    (4, (60000, 8192, 8193, 30000, 8192, 4096, 4097)),
])
def test_against_single_boxes(every, sizes):
    batch, boxes, alone, slots = Batch(), [], [], []
    for q, n in enumerate(sizes):
        prec = PRECISION_MIXED if q % 2 else PRECISION_FP64
        boxes.append(box(n, q + 1, prec))
        alone.append(box(n, q + 1, prec))
        slots.append(batch.attach(boxes[q], 9, 0.004, 1.0, 1.0, RCUT, SKIN, precision=prec, rebuild_every=every))
    while batch.step(9):
        pass
    for q, (b, c) in enumerate(zip(boxes, alone)):
        batch.detach(slots[q])
        c.run(9, 0.004, 1.0, 1.0, RCUT, SKIN, precision=PRECISION_MIXED if q % 2 else PRECISION_FP64, rebuild_every=every)
        eb, ec = b.export(), c.export()
        for k in ("cell", "id", "r", "v", "f", "ep"):
            assert np.array_equal(eb[k].view(np.uint8), ec[k].view(np.uint8)), (q, k)
