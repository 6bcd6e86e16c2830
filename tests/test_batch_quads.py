"""Batches on either side of the four-lanes-an-atom rules (by the batch's atoms) against the same
boxes run alone, bit for bit."""
import numpy as np
import pytest

from exanbody_amd import PRECISION_FP64, PRECISION_MIXED, Batch, Box, cubic_domain, generate_fcc

pytestmark = pytest.mark.gpu

RCUT, SKIN, STEPS = 2.5, 0.3, 23


def box(n, seed, precision):
    ncell = max(2, int(np.ceil((n / 4.0) ** (1.0 / 3.0) - 1e-9)))
    r, v, ids, length = generate_fcc(ncell, 0.8, n_atoms=n, jitter=0.02, temperature=1.2, seed=seed)
    d = cubic_domain(length, RCUT + SKIN)
    b = Box(d["bounds_min"], d["bounds_max"], d["grid_dims"], d["cell_size"])
    b.nbh_dist(RCUT, SKIN)
    b.set_particles(r, v, ids)
    b.init(1.0, 1.0, RCUT, SKIN, precision)
    return b


# all four lanes; small bricks with one lane; small and large bricks in one batch
@pytest.mark.parametrize("sizes", [(500, 3000, 867, 9000), (30000, 700, 20001), (60000, 55000, 900, 40000)])
@pytest.mark.parametrize("every", [10, 0])
@pytest.mark.parametrize("kinds", [(PRECISION_FP64,), (PRECISION_MIXED,), (PRECISION_FP64, PRECISION_MIXED)])
def test_against_single_boxes(sizes, every, kinds):
    prec = [kinds[q % len(kinds)] for q in range(len(sizes))]
    batch, boxes, alone = Batch(), [], []
    for q, n in enumerate(sizes):
        boxes.append(box(n, q + 1, prec[q]))
        alone.append(box(n, q + 1, prec[q]))
    steps = [STEPS - q for q in range(len(sizes))]  # they end one after another
    slots = [batch.attach(b, steps[q], 0.004, 1.0, 1.0, RCUT, SKIN, precision=prec[q], rebuild_every=every) for q, b in enumerate(boxes)]
    while batch.step(STEPS):
        pass
    for q, (b, c) in enumerate(zip(boxes, alone)):
        batch.detach(slots[q])
        c.run(steps[q], 0.004, 1.0, 1.0, RCUT, SKIN, precision=prec[q], rebuild_every=every)
        eb, ec = b.export(ghosts=True), c.export(ghosts=True)
        for k in ("cell", "id", "r", "v"):
            np.testing.assert_array_equal(eb[k].view(np.uint8), ec[k].view(np.uint8), err_msg=f"box {q}: {k}")
        eb, ec = b.export(), c.export()
        for k in ("f", "ep"):
            np.testing.assert_array_equal(eb[k].view(np.uint8), ec[k].view(np.uint8), err_msg=f"box {q}: {k}")
