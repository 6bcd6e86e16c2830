"""Four lanes an atom (small boxes' builds and LJ forces) against one lane an atom, bit for bit:
lists, forces, energies, trajectories."""
import numpy as np
import pytest

from exanbody_amd import PRECISION_FP64, PRECISION_MIXED, Box, cubic_domain
from exanbody_amd.workloads import lorentz_berthelot, slab_droplets

pytestmark = pytest.mark.gpu

RCUT, SKIN = 2.5, 0.3


def box(r, v, length, lanes, monkeypatch, bricks="2,2,1", types=None, rcut=RCUT, periodic=(1, 1, 1)):
    monkeypatch.setenv("XNB_BRICKS", f"{bricks},{lanes}")
    d = cubic_domain(length, rcut + SKIN)
    b = Box(d["bounds_min"], d["bounds_max"], d["grid_dims"], d["cell_size"], periodic=periodic)
    b.nbh_dist(rcut, SKIN)
    b.set_particles(r, v, None, types)
    return b


def same(a, c, keys=("cell", "id", "r", "v", "f", "ep")):
    ea, ec = a.export(ghosts=True), c.export(ghosts=True)
    for k in keys:
        np.testing.assert_array_equal(ea[k].view(np.uint8), ec[k].view(np.uint8), err_msg=k)


def same_streams(a, c):
    (sa, ma), (sc, mc) = a.streams(), c.streams()
    assert ma == mc
    np.testing.assert_array_equal(np.concatenate(sa), np.concatenate(sc))


def fluid(n, rho, seed):
    """n atoms on jittered simple cubic sites (no pair closer than 0.7), the last ones left out."""
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1.0 / 3.0) - 1e-9))
    a = rho ** (-1.0 / 3.0)
    q = rng.permutation(m ** 3)[:n]
    r = (np.stack([q % m, q // m % m, q // (m * m)], 1) + 0.5 + rng.uniform(-0.12, 0.12, (n, 3))) * a
    return r, rng.standard_normal((n, 3)), max(m * a, 2 * (RCUT + SKIN))


# a wave holds 16 atoms, a workgroup 64 or more; one atom, partly filled waves, several bricks
@pytest.mark.parametrize("precision", [PRECISION_FP64, PRECISION_MIXED])
@pytest.mark.parametrize("n,rho,bricks", [(1, 0.8, "1,1,1"), (2, 0.8, "2,1,1"), (17, 0.3, "1,1,1"), (500, 0.8, "1,1,1"),
                                          (513, 0.8, "2,2,2"), (1331, 0.5, "2,2,1"), (6859, 0.9, "2,2,2"), (4096, 1.3, "1,1,1")])
def test_run(n, rho, bricks, precision, monkeypatch):
    r, v, length = fluid(n, rho, n)
    a, c = (box(r, v, length, q, monkeypatch, bricks) for q in (1, 4))
    for b in (a, c):
        b.init(1.0, 1.0, RCUT, SKIN, precision)
    same(a, c)
    same_streams(a, c)
    for every, steps in ((5, 12), (0, 9)):
        ra, rc = (b.run(steps, 0.002, 1.0, 1.0, RCUT, SKIN, precision=precision, rebuild_every=every) for b in (a, c))
        assert ra == rc
        np.testing.assert_array_equal(a.run_step_counts(), c.run_step_counts())
        same(a, c)
    for b in (a, c):
        b.zero_particle_force()
        b.lennard_jones_force(0.7, 1.05, 2.3, precision=precision)
    same(a, c)


def test_lists_past_the_first_capacity_and_coincident_atoms(monkeypatch):
    """Density 2.2: up to about 200 neighbours against a first capacity of 96; two atoms on
    one point and two 1e-200 apart (the FP64 sums are walked again with the generic operations)."""
    r, v, length = fluid(4096, 2.2, 5)
    r[7], r[9] = r[11], 0.0
    r[13] = (1e-200, 0.0, 0.0)
    a, c = (box(r, v, length, q, monkeypatch, "1,1,1") for q in (1, 4))
    for b in (a, c):
        b.init(1.0, 1.0, RCUT, SKIN, PRECISION_FP64)
    same_streams(a, c)
    ea, ec = a.export(), c.export()
    for k in ("f", "ep"):
        nan = np.isnan(ea[k])
        np.testing.assert_array_equal(nan, np.isnan(ec[k]))
        np.testing.assert_array_equal(ea[k][~nan].view(np.uint64), ec[k][~nan].view(np.uint64))


def test_parameters_the_fast_pair_does_not_cover(monkeypatch):
    r, v, length = fluid(700, 0.8, 3)
    a, c = (box(r, v, length, q, monkeypatch) for q in (1, 4))
    for b in (a, c):
        b.init(1.0, 1.0, RCUT, SKIN, PRECISION_FP64)
        b.zero_particle_force()
        b.lennard_jones_force(1.0, 1e120, RCUT)
    ea, ec = a.export(), c.export()
    np.testing.assert_array_equal(np.isnan(ea["f"]), np.isnan(ec["f"]))


@pytest.mark.parametrize("precision", [PRECISION_FP64, PRECISION_MIXED])
def test_other_forces_on_quad_lists(precision, monkeypatch):
    """The multi-material and gravitational forces read these lists with one lane an atom; a
    multi-material run builds them with each type pair's radius."""
    r, v, _, types, d = slab_droplets(n_atoms=26364, ncell=26, n_droplets=6, seed=4)
    eps, sig, rc = lorentz_berthelot()
    out = []
    for lanes in (1, 4):
        monkeypatch.setenv("XNB_BRICKS", f"1,1,1,{lanes}")
        b = Box(d["bounds_min"], d["bounds_max"], d["grid_dims"], d["cell_size"], periodic=d["periodic"])
        b.nbh_dist(float(rc.max()), SKIN)
        b.set_particles(r, v, None, types)
        b.init(1.0, 1.0, float(rc.max()), SKIN, precision)
        b.run_multimat(12, 0.002, 2, eps, sig, rc, SKIN, precision=precision, rebuild_every=5)
        b.gravitational_force(0.5, [1.0, 2.0], 2.0)
        out.append(b)
    same(*out)
    same_streams(*out)
