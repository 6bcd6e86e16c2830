"""A destroyed box gives back all the device memory it held."""
import ctypes as C

import pytest

from exanbody_amd import PRECISION_FP64, Batch, load
from tests.helpers import RCUT, SKIN, fcc_inputs, make_pair

pytestmark = pytest.mark.gpu


def _free_bytes():
    load()
    hip = C.CDLL("libamdhip64.so.7")  # the runtime the library has loaded
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


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
    free = _free_bytes()
    for _ in range(12):
        assert _use(batched) > 20 << 20
    assert free - _free_bytes() < 6 << 20, held
