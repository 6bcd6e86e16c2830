"""A destroyed box gives back all the device memory it held."""
import pytest
import torch

from exanbody_amd import PRECISION_FP64, Batch
from tests.helpers import RCUT, SKIN, fcc_inputs, make_pair

pytestmark = pytest.mark.gpu


def _use(batched):
    r, v, ids, L = fcc_inputs(23, temperature=1.0, seed=3)  # 48,668 atoms
    _, b, _ = make_pair(r, v, ids, L)
    b.init(1.0, 1.0, RCUT, SKIN, PRECISION_FP64)
    if batched:
        B = Batch()
        slot = B.attach(b, 3, 0.002, 1.0, 1.0, RCUT, SKIN, rebuild_every=2)
        while B.step(3):
            pass
        B.detach(slot)
        B.close()
    else:
        b.run(3, 0.002, 1.0, 1.0, RCUT, SKIN, rebuild_every=2)
    b.streams()
    b.energies()
    held, _ = b.device_bytes()
    b.close()
    return held


@pytest.mark.parametrize("batched", [False, True])
def test_destroyed_boxes_leave_no_device_memory(batched):
    """Twelve boxes one after another: each holds tens of megabytes, and an array of 4 bytes per
    region atom left behind by each (about a megabyte) would show."""
    held = _use(batched)
    free, _ = torch.cuda.mem_get_info()
    for _ in range(12):
        assert _use(batched) > 20 << 20
    assert free - torch.cuda.mem_get_info()[0] < 6 << 20, held
