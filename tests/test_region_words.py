"""The force's staging words: ghosts placed by their sources in runs, by their own (possibly stale)
slots in operators, against the oracle bit for bit; bricks from one atom to a full workgroup."""
import numpy as np
import pytest

from exanbody_amd import PRECISION_FP64, Box, cubic_domain
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

RCUT, SKIN = 2.5, 0.3


def pair_of(n, rho, seed, bricks, monkeypatch):
    if bricks:
        monkeypatch.setenv("XNB_BRICKS", bricks)
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1.0 / 3.0) - 1e-9))
    a = rho ** (-1.0 / 3.0)
    q = rng.permutation(m ** 3)[:n]
    r = (np.stack([q % m, q // m % m, q // (m * m)], 1) + 0.5 + rng.uniform(-0.12, 0.12, (n, 3))) * a
    v = rng.standard_normal((n, 3))
    d = cubic_domain(max(m * a, 2 * (RCUT + SKIN)), RCUT + SKIN)
    ids = np.arange(n, dtype=np.uint64)
    o = Oracle(d["bounds_min"], d["bounds_max"], d["grid_dims"], d["cell_size"], ghost_dist=RCUT + SKIN)
    o.set_particles(r, v, ids)
    o.init(1.0, 1.0, RCUT, SKIN)
    b = Box(d["bounds_min"], d["bounds_max"], d["grid_dims"], d["cell_size"])
    b.nbh_dist(RCUT, SKIN)
    b.set_particles(r, v, ids)
    b.init(1.0, 1.0, RCUT, SKIN, PRECISION_FP64)
    return o, b


def same(o, b, keys=("r", "v", "f"), ghosts=False):
    eo, eb = o.export(ghosts=ghosts), b.export(ghosts=ghosts)
    np.testing.assert_array_equal(eo["id"], eb["id"])
    for k in keys:
        np.testing.assert_array_equal(np.ascontiguousarray(eo[k]).view(np.uint64), np.ascontiguousarray(eb[k]).view(np.uint64), err_msg=k)


# 1 atom; bricks of a few atoms; one and four lanes an atom; a region of more than one staging round
@pytest.mark.parametrize("n,rho,bricks", [(1, 0.8, ""), (40, 0.3, "1,1,1,1"), (900, 0.8, ""), (900, 0.8, "4,4,2,1"),
                                          (4913, 0.85, "1,1,1,4"), (4913, 0.85, "1,1,1,1"), (9261, 0.8, "4,2,2,1")])
def test_runs_then_operators(n, rho, bricks, monkeypatch):
    o, b = pair_of(n, rho, n, bricks, monkeypatch)
    for steps in (7, 5):  # ends between rebuilds, then over one
        o.run(steps, 0.002, 1.0, 1.0, RCUT, SKIN, rebuild_every=10)
        b.run(steps, 0.002, 1.0, 1.0, RCUT, SKIN, precision=PRECISION_FP64, rebuild_every=10)
        same(o, b)
        same(o, b, keys=("r",), ghosts=True)
        # moved atoms, ghosts where they were: an operator's force reads them there
        o.push_f_v_r(0.004)
        b.push_f_v_r(0.004)
        for _ in range(2):
            o.zero_force()
            o.lj_force(1.0, 1.0, RCUT)
            b.zero_particle_force()
            b.lennard_jones_force(1.0, 1.0, RCUT)
            same(o, b)
            o.ghost_update_r()
            b.ghost_update_r()


def test_other_forces_read_stale_ghosts(monkeypatch):
    o, b = pair_of(2744, 0.8, 3, "", monkeypatch)
    o.run(3, 0.002, 1.0, 1.0, RCUT, SKIN, rebuild_every=10)
    b.run(3, 0.002, 1.0, 1.0, RCUT, SKIN, precision=PRECISION_FP64, rebuild_every=10)
    o.push_f_v_r(0.004)
    b.push_f_v_r(0.004)
    o.zero_force()
    b.zero_particle_force()
    o.gravitational_force(0.5, [1.5], 2.0)
    b.gravitational_force(0.5, [1.5], 2.0)
    same(o, b)
    o.zero_force()
    b.zero_particle_force()
    o.lj_force_multimat(1, [1.0], [1.0], [RCUT])
    b.lennard_jones_force_multimat(1, [1.0], [1.0], [RCUT])
    same(o, b)
    # and a run after them places ghosts by their sources again
    o.run(4, 0.002, 1.0, 1.0, RCUT, SKIN, rebuild_every=0)
    b.run(4, 0.002, 1.0, 1.0, RCUT, SKIN, precision=PRECISION_FP64, rebuild_every=0)
    same(o, b)
