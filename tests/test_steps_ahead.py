"""Runs on the displacement trigger, whose steps are launched ahead of the host's look at their
counts, against the same steps run one at a time: state, rebuilds and step counts bit for bit."""
import numpy as np
import pytest

from exanbody_amd import PRECISION_FP64, PRECISION_MIXED, Box, cubic_domain, generate_fcc
from exanbody_amd.workloads import lorentz_berthelot, slab_droplets

pytestmark = pytest.mark.gpu

RCUT, SKIN = 2.5, 0.3


def same(a, b):
    ea, eb = a.export(ghosts=True), b.export(ghosts=True)
    for k in ("cell", "id", "r", "v", "f", "ep"):
        np.testing.assert_array_equal(ea[k].view(np.uint8), eb[k].view(np.uint8), err_msg=k)


# rebuilds in nearly every step (hot), every few steps, and none at all (cold); runs that end
# before, on and after the first rebuild; 4,000 atoms: quads, 108,000: one lane an atom
@pytest.mark.parametrize("precision", [PRECISION_FP64, PRECISION_MIXED])
@pytest.mark.parametrize("ncell,temperature,dt", [(10, 60.0, 0.004), (10, 1.0, 0.005), (10, 1e-6, 0.001), (30, 1.5, 0.005)])
@pytest.mark.parametrize("steps", [1, 2, 33])
def test_against_single_steps(ncell, temperature, dt, steps, precision):
    r, v, ids, length = generate_fcc(ncell, 0.8442, jitter=0.02, temperature=temperature, seed=5)
    d = cubic_domain(length, RCUT + SKIN)
    boxes = []
    for _ in range(2):
        b = Box(d["bounds_min"], d["bounds_max"], d["grid_dims"], d["cell_size"])
        b.nbh_dist(RCUT, SKIN)
        b.set_particles(r, v, ids)
        b.init(1.0, 1.0, RCUT, SKIN, precision)
        boxes.append(b)
    a, b = boxes
    b.timer_enable(True)  # timed runs look at every step's count before the next
    kw = dict(precision=precision, rebuild_every=0)
    for _ in range(2):
        ra = a.run(steps, dt, 1.0, 1.0, RCUT, SKIN, **kw)
        rb = b.run(steps, dt, 1.0, 1.0, RCUT, SKIN, **kw)
        assert ra == rb
        np.testing.assert_array_equal(a.run_step_counts(), b.run_step_counts())
        same(a, b)


def test_multimat():
    r, v, _, types, d = slab_droplets(n_atoms=26364, ncell=26, n_droplets=6, seed=4)
    eps, sig, rc = lorentz_berthelot()
    boxes = []
    for timed in (False, True):
        b = Box(d["bounds_min"], d["bounds_max"], d["grid_dims"], d["cell_size"], periodic=d["periodic"])
        b.nbh_dist(float(rc.max()), SKIN)
        b.set_particles(r, v, None, types)
        b.init(1.0, 1.0, float(rc.max()), SKIN, PRECISION_FP64)
        b.timer_enable(timed)
        b.run_multimat(40, 0.004, 2, eps, sig, rc, SKIN, precision=PRECISION_FP64, rebuild_every=0)
        boxes.append(b)
    same(*boxes)
